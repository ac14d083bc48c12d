"""The large copies to the host (yrh_stage.hip) on a stand-in for the HIP
runtime that copies at once and keeps the rules the real one has: an event can
only be recorded on a stream of the device that was current when the event was
made. Covers what one GPU cannot show: another current device, destinations
that are not pageable, a host out of threads or memory."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

pytestmark = pytest.mark.skipif(shutil.which("g++") is None, reason="g++ not available")

PROGRAM = r"""
#include "yrh_internal.h"

#include <atomic>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <new>
#include <vector>

// ---- the stand-in runtime: streams and events are the number of their device + 1
static thread_local int current = 0;
static hipMemoryType kind = hipMemoryTypeUnregistered;
static bool pinned_fails = false;
static std::atomic<int> live_threads{1};
static std::atomic<long> copies{0};
extern "C" {
hipError_t hipSetDevice(int d) { current = d; return hipSuccess; }
hipError_t hipGetDevice(int* d) { *d = current; return hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) { *e = (hipEvent_t)(size_t)(current + 1); return hipSuccess; }
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t e, hipStream_t s) {
    return (size_t)e == (size_t)s ? hipSuccess : hipErrorInvalidHandle;
}
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipHostMalloc(void** p, size_t n, unsigned) {
    if (pinned_fails) return hipErrorOutOfMemory;
    *p = std::malloc(n);
    return hipSuccess;
}
hipError_t hipHostFree(void* p) { std::free(p); return hipSuccess; }
hipError_t hipFree(void*) { return hipSuccess; }
hipError_t hipGetLastError() { return hipSuccess; }
const char* hipGetErrorString(hipError_t) { return "error"; }
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind, hipStream_t) {
    ++copies;
    std::memcpy(d, s, n);
    return hipSuccess;
}
hipError_t hipPointerGetAttributes(hipPointerAttribute_t* a, const void*) {
    std::memset(a, 0, sizeof(*a));
    a->type = kind;
    return hipSuccess;
}
int roctxRangePushA(const char*) { return 0; }
int roctxRangePop() { return 0; }
}
namespace yrh {
int Fail(yrh_context* ctx, int code, const std::string& m) { ctx->error = m; return code; }
int CheckHip(yrh_context* ctx, hipError_t e, const char* what) { return e == hipSuccess ? YRH_OK : Fail(ctx, YRH_E_HIP, what); }
}

// Allocations of this thread before one fails (-1: none does).
static thread_local int allocations_left = -1;
void* operator new(size_t n) {
    if (allocations_left == 0) throw std::bad_alloc();
    if (allocations_left > 0) --allocations_left;
    return std::malloc(n ? n : 1);
}
void* operator new(size_t n, const std::nothrow_t&) noexcept {
    if (allocations_left == 0) return nullptr;
    if (allocations_left > 0) --allocations_left;
    return std::malloc(n ? n : 1);
}
void operator delete(void* p) noexcept { std::free(p); }
void operator delete(void* p, size_t) noexcept { std::free(p); }

static const size_t MIB = size_t{1} << 20;
static std::vector<unsigned char> src, dst;

// Copies n bytes; whether it was taken. Every byte of a taken copy must arrive, none beyond it.
static bool Copy(yrh_context& ctx, size_t n, int fail_after = -1) {
    std::memset(dst.data(), 7, n + 64);
    bool done = false;
    allocations_left = fail_after;
    const int rc = yrh::StagedCopyToHost(&ctx, dst.data(), src.data(), n, &done);
    allocations_left = -1;
    if (rc != YRH_OK) { std::printf("copy of %zu bytes failed: %s\n", n, ctx.error.c_str()); std::exit(1); }
    if (done && std::memcmp(dst.data(), src.data(), n) != 0) { std::printf("copy of %zu bytes: wrong bytes\n", n); std::exit(1); }
    for (size_t k = done ? n : 0; k < n + 64; ++k) {
        if (dst[k] != 7) { std::printf("copy of %zu bytes wrote past its end\n", n); std::exit(1); }
    }
    return done;
}

#define EXPECT(x) do { if (!(x)) { std::printf("line %d: %s\n", __LINE__, #x); std::exit(1); } } while (0)

static void Open(yrh_context& ctx, int device) {
    ctx.device = device;
    ctx.stream = (hipStream_t)(size_t)(device + 1);
}

int main(int argc, char** argv) {
    const std::string what = argv[1];
    src.resize(48 * MIB);
    dst.resize(48 * MIB + 64);
    for (size_t k = 0; k < src.size(); ++k) src[k] = (unsigned char)(k * 2654435761u >> 13);
    if (what == "sizes") {
        yrh_context ctx;
        Open(ctx, 0);
        EXPECT(!Copy(ctx, 8 * MIB));  // a context's first, under 32 MiB
        const size_t sizes[] = {6 * MIB, 6 * MIB + 1, 7 * MIB + 4093, 9 * MIB + 1, 11 * MIB, 13 * MIB - 1, 15 * MIB + 1,
                                16 * MIB, 17 * MIB + 1, 32 * MIB, 41 * MIB + 7};
        for (size_t n : sizes) EXPECT(Copy(ctx, n));
        EXPECT(!Copy(ctx, 6 * MIB - 1));
        EXPECT(!Copy(ctx, 1));
        yrh::DestroyHostStage(&ctx);
        Open(ctx, 0);
        ctx.large_copy_seen = false;
        EXPECT(Copy(ctx, 32 * MIB));  // a context's first
        yrh::DestroyHostStage(&ctx);
    } else if (what == "device") {
        // The caller works on device 0, the context is on device 1.
        yrh_context ctx;
        Open(ctx, 1);
        current = 0;
        EXPECT(Copy(ctx, 40 * MIB));
        EXPECT(current == 0);
        EXPECT(Copy(ctx, 9 * MIB));
        EXPECT(current == 0);
        yrh::DestroyHostStage(&ctx);
    } else if (what == "memory") {
        yrh_context ctx;
        Open(ctx, 0);
        for (hipMemoryType k : {hipMemoryTypeHost, hipMemoryTypeDevice, hipMemoryTypeManaged}) {
            kind = k;
            EXPECT(!Copy(ctx, 40 * MIB));
        }
        EXPECT(ctx.stage == nullptr);
        kind = hipMemoryTypeUnregistered;
        EXPECT(Copy(ctx, 40 * MIB));
        kind = hipMemoryTypeHost;
        EXPECT(!Copy(ctx, 40 * MIB));
        yrh::DestroyHostStage(&ctx);
    } else {
        // Pinned memory, then each host allocation of a copy in turn, cannot be had.
        yrh_context ctx;
        Open(ctx, 0);
        pinned_fails = true;
        EXPECT(!Copy(ctx, 40 * MIB));
        pinned_fails = false;
        EXPECT(!Copy(ctx, 40 * MIB, 0));
        EXPECT(Copy(ctx, 40 * MIB));
        for (int k = 0; k < 12; ++k) EXPECT(Copy(ctx, 40 * MIB, k));
        yrh::DestroyHostStage(&ctx);
    }
    std::printf("ok\n");
}
"""


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    d = tmp_path_factory.mktemp("stage")
    (d / "main.cpp").write_text(PROGRAM)
    flags = ["-std=c++17", "-O1", "-w", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
             "-I" + os.path.join(ROOT, "yaoray_amd", "csrc"), "-I" + os.path.join(ROOT, "include")]
    subprocess.run(["g++", *flags, "-x", "c++", os.path.join(ROOT, "yaoray_amd", "csrc", "yrh_stage.hip"),
                    str(d / "main.cpp"), "-lpthread", "-o", str(d / "stage")], check=True)
    return str(d / "stage")


@pytest.mark.parametrize("what", ["sizes", "device", "memory", "failures"])
def test_staged_copy(program, what):
    r = subprocess.run([program, what], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0 and r.stdout == "ok\n", r.stdout + r.stderr
