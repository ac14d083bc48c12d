// BVH traversal for MI355X (gfx950): the closest-hit / any-hit machinery
// shared by the ray-cast kernels (yrh_trace.hip) and the render kernels that
// trace inside a longer per-ray loop (yrh_render.hip).
//
// Arithmetic follows the reference operation by operation, with FP
// contraction disabled (the reference x86-64 build has no FMA):
//   slab test      include/yaoray/core/bounds.hpp:50-90
//   triangle test  src/accel/bvh_traversal.cpp:52-121 (Moller-Trumbore, two-sided,
//                  |det| < 1e-8 reject, equal-t tie -> lower flat triangle index)
//   traversal      src/accel/bvh_traversal.cpp:253-345 (root box, pop-skip when
//                  entry_t > best t, both child boxes, push far then near, ties
//                  near = left)
//   two-level      src/accel/two_level_bvh.cpp:365-481 (object ray through the
//                  host inverse, unnormalised direction so t is shared, BLAS run
//                  with t_max = best t, accepted only if strictly closer)
// so hit ids, t, barycentrics and the node/triangle test counters equal the
// reference's on the same tree.
//
// Execution model: a persistent grid sized to the device. Each wave64 refills
// idle lanes from a global ray counter with one atomic per wave (ballot +
// mbcnt), so divergent ray lengths do not idle the wave. A lane's next record
// is one register (`cur`: an interior node, a primitive slot, an instance
// slot, or none); the stack holds the far siblings only, in LDS (the first
// lds_levels entries per lane, a launch option up to kMaxLdsStack; laid out
// [wave][level][lane] so a wave's pushes hit consecutive banks) and deeper
// levels in a per-lane global region; one pending sibling per level fits its
// capacity, max_depth + 2.
//
// What bounds it: instruction issue (VALU busy 0.94 with 0.37 of the lanes
// active for 8.39 M rays on 1 M triangles, 1.0 and 0.25 for the instanced 1080p
// frame) and, as much, the lanes' own 16-byte record requests (TD busy 0.95 and
// 0.94). One-register records, an end-of-leaf mark in the slot, constant-stride
// stack addresses and no per-rejection branches in the triangle test took the
// 1 M-triangle cast from 4.15 to 3.81 ms a call, 1.29 M rays on 2000 instances
// from 437 to 333 us (three contexts' calls in flight), the frame at 16 spp from
// 190 to 144 ms.
//
// A policy object supplies each ray's first segment (Begin) and receives each
// finished segment with its origin and direction (Finish); Finish may hand
// back a further segment of the same ray, which the lane traverses next
// without giving up its slot. The plain ray-cast policy writes the hit and
// ends the ray; the transparent-shadow policy walks a shadow ray through
// dielectric surfaces this way.
#pragma once

#include "yrh_internal.h"

#pragma clang fp contract(off)

namespace yrh {
namespace trav {

constexpr int kMaxLdsStack = 16;  // LDS stack levels per lane, at most (launch option)
constexpr int kMaxBlock = 256;
constexpr int kRefillIdleLanes = 32;  // refill once half the wave is idle (swept: 8..56)
constexpr int kParts = 8;             // claim ranges, one per XCD
constexpr int kPartStride = 32;       // words between their counters: one cache line each
// Test sums are kept in copies on cache lines of their own; workgroup b adds
// to copy b % kTotalsSlots. On one line the 4096 waves of a bounce took 228 us
// to add theirs, however few rays they had traced.
constexpr int kTotalsSlots = 64;
constexpr int kTotalsStride = 16;

struct TraceArgs {
    const float4* org;
    const float4* dir;
    int32_t n;
    const uint32_t* n_device;    // when set, the ray count is read from device memory
    // optional test sums: kTotalsSlots copies kTotalsStride words apart, each
    // [0] node, [1] triangle, [2] sphere tests
    unsigned long long* totals;
    // outputs
    float4* hit;
    int32_t* inst_out;
    uint32_t* node_tests;
    uint32_t* triangle_tests;
    uint32_t* sphere_tests;
    uint32_t* occluded;
    // flat BVH, or BLASes and TLAS (yrh_internal.h)
    const float4* arena;
    int32_t root_code;
    float root_lo_x, root_lo_y, root_lo_z, root_hi_x, root_hi_y, root_hi_z;
    int32_t empty;
    // scheduling
    uint32_t* counter;       // this launch's kParts ray counters, kPartStride words apart (zero at launch)
    uint32_t* next_counter;  // the next launch's counters, zeroed here (may be null)
    int32_t spread_waves;    // waves that a short queue is spread over
    const int32_t* order;    // claim position -> ray index (null = identity)
    uint32_t* overflow;      // stack overflow flag
    int2* spill;
    int64_t spill_stride;
    int32_t capacity;
    int32_t lds_levels;  // stack levels held in LDS (dynamic shared memory: lds_levels x block int2)
};

// Lanes for which `p` holds.
__device__ __forceinline__ uint64_t Ballot(bool p) { return __builtin_amdgcn_ballot_w64(p); }

// 1 / x, correctly rounded as the reference's division: two Newton steps in
// FMA on the hardware reciprocal (P. Markstein, "Computation of elementary
// functions on the IBM RISC System/6000 processor", 1990), 5 instructions
// against the 11 of the general division. Equal to it for every |x| in
// [2^-100, 2^100] (tests/test_trace_gpu.py: every mantissa at the ends of the
// range and in between); a wave with a lane outside (zero, infinite and NaN
// included) runs the general division too.
// `below`: values under 2^-100 occur (else their result is not used).
template <bool below>
__device__ __forceinline__ float Reciprocal(float x) {
    float r = __builtin_amdgcn_rcpf(x);
    r = __builtin_fmaf(__builtin_fmaf(-x, r, 1.0f), r, r);
    r = __builtin_fmaf(__builtin_fmaf(-x, r, 1.0f), r, r);
    const float ax = fabsf(x);
    const bool outside = below ? !(ax >= 0x1p-100f && ax <= 0x1p100f) : !(ax <= 0x1p100f);
    if (Ballot(outside) != 0) {
        const float general = 1.0f / x;
        r = outside ? general : r;
    }
    return r;
}

// The ray being traversed: its origin and direction reciprocals.
struct RayPre {
    float ox, oy, oz;
    float ix, iy, iz;
    bool nx, ny, nz;
};

__device__ __forceinline__ RayPre Precompute(float ox, float oy, float oz, float dx, float dy, float dz) {
    RayPre r;
    r.ox = ox;
    r.oy = oy;
    r.oz = oz;
    r.ix = Reciprocal<true>(dx);
    r.iy = Reciprocal<true>(dy);
    r.iz = Reciprocal<true>(dz);
    r.nx = signbit(r.ix);
    r.ny = signbit(r.iy);
    r.nz = signbit(r.iz);
    return r;
}

// IntersectBounds. The reference narrows the interval with comparisons
// (t_min = an > t_min ? an : t_min, t_max = af < t_max ? af : t_max), which
// keep the bound when a 0*inf product is NaN. fmaxf / fminf (IEEE maxNum /
// minNum, v_max3_f32 / v_min3_f32 here) return the same value for every
// input: a NaN operand yields the other operand, and the bounds themselves are
// never NaN; only the sign of a zero result may differ, which no comparison
// below can observe. Near / far planes are still chosen by direction sign, as
// the reference does, not by min / max of the two plane distances (that
// would differ on a NaN distance).
__device__ __forceinline__ bool Slab(const RayPre& r, float lx, float ly, float lz, float hx, float hy, float hz,
                                     float t_min, float t_max, float& entry) {
    const float anx = ((r.nx ? hx : lx) - r.ox) * r.ix;
    const float afx = ((r.nx ? lx : hx) - r.ox) * r.ix;
    const float any = ((r.ny ? hy : ly) - r.oy) * r.iy;
    const float afy = ((r.ny ? ly : hy) - r.oy) * r.iy;
    const float anz = ((r.nz ? hz : lz) - r.oz) * r.iz;
    const float afz = ((r.nz ? lz : hz) - r.oz) * r.iz;
    t_min = fmaxf(fmaxf(anx, any), fmaxf(anz, t_min));
    t_max = fminf(fminf(afx, afy), fminf(afz, t_max));
    entry = t_min;
    return t_max >= t_min;
}

// The closest hit so far. u holds kNoHitU until there is one: every id is a
// valid hit (flat triangle indices come from the caller, -1 among them), and an
// accepted triangle's u is at least 0 or NaN, a sphere's never near -1.
constexpr float kNoHitU = -1.0f;
struct Best {
    float t;
    float u;
    float v;
    int32_t id;
    static __device__ __forceinline__ Best None(float t) { return Best{t, kNoHitU, 0.0f, -1}; }
    __device__ __forceinline__ bool Hit() const { return u != kNoHitU; }
    // The hit record: (t, u, v, id), u = v = 0 and id = -1 without a hit.
    __device__ __forceinline__ float4 Record() const {
        return make_float4(t, Hit() ? u : 0.0f, v, __int_as_float(id));
    }
};

// IntersectTriangle on a (p0, e1, e2) slot. Returns true when `best` changed.
// Every rejection of the reference is one term of the final condition: with a
// dozen lanes of a wave in here, some lane passes each of them, so skipping
// ahead would only add mask bookkeeping.
template <bool kAny>
__device__ __forceinline__ bool TriangleTest(const float4& s0, const float4& s1, const float4& s2,
                                             float ox, float oy, float oz, float dx, float dy, float dz,
                                             float t_min, Best& best) {
    const float e1x = s1.x, e1y = s1.y, e1z = s1.z;
    const float e2x = s2.x, e2y = s2.y, e2z = s2.z;
    // pvec = Cross(d, e2)
    const float px = dy * e2z - dz * e2y;
    const float py = dz * e2x - dx * e2z;
    const float pz = dx * e2y - dy * e2x;
    const float det = e1x * px + e1y * py + e1z * pz;
    const float inv_det = Reciprocal<false>(det);
    const float tx = ox - s0.x;
    const float ty = oy - s0.y;
    const float tz = oz - s0.z;
    const float u = (tx * px + ty * py + tz * pz) * inv_det;
    // qvec = Cross(tvec, e1)
    const float qx = ty * e1z - tz * e1y;
    const float qy = tz * e1x - tx * e1z;
    const float qz = tx * e1y - ty * e1x;
    const float v = (dx * qx + dy * qy + dz * qz) * inv_det;
    const float t = (e2x * qx + e2y * qy + e2z * qz) * inv_det;
    const int32_t id = __float_as_int(s0.w);
    // Rejections in the reference's form: a NaN passes them as it does there.
    bool reject = (fabsf(det) < 1.0e-8f) | (u < 0.0f) | (u > 1.0f) | (v < 0.0f) | (u + v > 1.0f) | (t <= t_min) |
                  (t > best.t);
    // Equal t: the lower flat index stays (a sphere or no hit, negative, never does).
    if (!kAny) reject |= (t == best.t) & (best.id >= 0) & (id >= best.id);
    if (reject) return false;
    best.t = t;
    best.id = id;
    best.u = u;
    best.v = v;
    return true;
}

// Sphere slot of a leaf (device layout): (centre, id bits) (radius, 0, 0, last)
// (0, 0, 0, 0) with id = -2 - sphere index; triangle slots carry their flat
// triangle index (>= 0) in the same word.
__device__ __forceinline__ bool IsSphereId(int32_t id) { return id <= -2; }

// SphereUv (src/geometry/intersection.cpp:136-151) of the outward normal at
// ray.At(t): the (u, v) the reference stores in a sphere hit.
__device__ __forceinline__ void SphereUv(float cx, float cy, float cz, float ox, float oy, float oz, float dx, float dy,
                                         float dz, float t, float& u, float& v) {
    const float px = ox + dx * t, py = oy + dy * t, pz = oz + dz * t;
    const float nx = px - cx, ny = py - cy, nz = pz - cz;
    const float len = sqrtf(nx * nx + ny * ny + nz * nz);
    float n0 = 0.0f, n1 = 0.0f, n2 = 0.0f;
    if (len > 0.0f) {
        n0 = nx / len;
        n1 = ny / len;
        n2 = nz / len;
    }
    constexpr float kPi = 3.14159265358979323846f;
    const float y = fminf(fmaxf(n1, -1.0f), 1.0f);
    u = (atan2f(n0, n2) + kPi) / (2.0f * kPi);
    v = (kPi - acosf(y)) / kPi;
}

// IntersectAnalyticSphere (src/accel/bvh_traversal.cpp:123-150) over
// IntersectSphere (src/geometry/intersection.cpp:108-128), same operations in
// the same order: the nearer root if it lies in (t_min, best t), else the
// farther one; a hit is strictly closer than `best` and clears the triangle
// id. (u, v) = SphereUv when `with_uv` (ray casts report it; renders
// recompute the normal). Returns true when `best` changed.
__device__ __forceinline__ bool SphereTest(float cx, float cy, float cz, float radius, int32_t id, float ox, float oy,
                                           float oz, float dx, float dy, float dz, float t_min, bool with_uv,
                                           Best& best) {
    const float ocx = ox - cx, ocy = oy - cy, ocz = oz - cz;
    const float a = dx * dx + dy * dy + dz * dz;
    const float b = 2.0f * (ocx * dx + ocy * dy + ocz * dz);
    const float c = (ocx * ocx + ocy * ocy + ocz * ocz) - radius * radius;
    const float disc = b * b - 4.0f * a * c;
    if (disc < 0.0f) return false;
    const float sq = sqrtf(disc);
    const float inv_2a = 0.5f / a;
    float t = (-b - sq) * inv_2a;
    if (!(t > t_min && t < best.t)) {
        t = (-b + sq) * inv_2a;
        if (!(t > t_min && t < best.t)) return false;
    }
    best.t = t;
    best.id = id;
    best.u = 0.0f;
    best.v = 0.0f;
    if (with_uv) SphereUv(cx, cy, cz, ox, oy, oz, dx, dy, dz, t, best.u, best.v);
    return true;
}

// LDS word of the traversal stack, in the LDS address space so that its
// stores stay ds_write (a generic pointer lets the compiler merge them with
// the spill stores into flat stores).
typedef __attribute__((address_space(3))) uint64_t LdsWord;
constexpr uint32_t kStackStep = 64 * sizeof(uint64_t);  // one level of a wave

// Per-lane traversal stack of (code, entry distance). `sp` is the LDS address
// of the next free entry, kStackStep per level; it runs on past `limit` for the
// levels in the global spill region, so a push or pop in LDS is one compare,
// one add and one LDS access (no multiplication by a run-time stride).
struct Stack {
    uint32_t base;   // this lane's column
    uint32_t limit;  // first address past its LDS levels
    uint32_t sp;
    int2* spill;  // this lane's column in the global spill region
    int64_t spill_stride;
    int32_t capacity;
    uint32_t* overflow;  // the launch's overflow flag

    __device__ __forceinline__ void Init(const TraceArgs& a, const int2* lds) {
        const int wave = static_cast<int>(threadIdx.x >> 6);
        const int lane = static_cast<int>(threadIdx.x & 63u);
        const int levels = a.lds_levels < a.capacity ? a.lds_levels : a.capacity;
        base = static_cast<uint32_t>(reinterpret_cast<uintptr_t>((const LdsWord*)(lds))) +
               static_cast<uint32_t>(wave * a.lds_levels) * kStackStep + static_cast<uint32_t>(lane) * sizeof(uint64_t);
        limit = base + static_cast<uint32_t>(levels) * kStackStep;
        sp = base;
        spill = a.spill + static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
        spill_stride = a.spill_stride;
        capacity = a.capacity;
        overflow = a.overflow;
    }
    __device__ __forceinline__ bool Empty() const { return sp == base; }
    __device__ __forceinline__ void Clear() { sp = base; }
    __device__ __forceinline__ int2* Spilled() const {
        return spill + static_cast<int64_t>((sp - limit) / kStackStep) * spill_stride;
    }
    __device__ __forceinline__ void Push(int32_t code, float entry) {
        if (sp < limit) {
            *reinterpret_cast<LdsWord*>(sp) = static_cast<uint64_t>(static_cast<uint32_t>(code)) |
                                              (static_cast<uint64_t>(__float_as_uint(entry)) << 32);
        } else if (static_cast<int32_t>((sp - base) / kStackStep) < capacity) {
            *Spilled() = make_int2(code, __float_as_int(entry));
        } else {
            atomicOr(overflow, 1u);  // dropped: the launch then fails
            sp -= kStackStep;
        }
        sp += kStackStep;
    }
    // The stack must not be empty.
    __device__ __forceinline__ void Pop(int32_t& code, float& entry) {
        sp -= kStackStep;
        if (sp < limit) {
            const uint64_t w = *reinterpret_cast<LdsWord*>(sp);
            code = static_cast<int32_t>(static_cast<uint32_t>(w));
            entry = __uint_as_float(static_cast<uint32_t>(w >> 32));
        } else {
            const int2 e = *Spilled();
            code = e.x;
            entry = __int_as_float(e.y);
        }
    }
};

// One interior step on a fetched node record (a, b, c = both child boxes,
// codes cl, cr): tests both boxes as the reference does and returns the
// nearer hit child (ties go left), the farther one pushed; kNoRecord when
// neither is hit. The reference pushes the near child too and pops it next:
// its entry is within the bound, so the pop always takes it.
__device__ __forceinline__ int32_t InteriorStep(const float4& na, const float4& nb, const float4& nc, int32_t cl,
                                                int32_t cr, const RayPre& r, float t_min, float t_max, Stack& st) {
    float el, er;
    const bool hl = Slab(r, na.x, na.y, na.z, na.w, nb.x, nb.y, t_min, t_max, el);
    const bool hr = Slab(r, nb.z, nb.w, nc.x, nc.y, nc.z, nc.w, t_min, t_max, er);
    const bool left = hl && (!hr || el <= er);
    if (hl && hr) st.Push(left ? cr : cl, left ? er : el);
    return left ? cl : (hr ? cr : kNoRecord);
}

// The record a lane fetches in one traversal iteration: a 64-byte node or a
// 48-byte primitive slot, loaded before either is processed, so a wave whose
// lanes are split between interior nodes and leaves waits for one memory
// latency per iteration instead of one per branch and per triangle.
struct Fetch {
    float4 q0, q1, q2;
    int2 q3;
    __device__ __forceinline__ void Load(const float4* p, bool node) {
        q0 = p[0];
        q1 = p[1];
        q2 = p[2];
        if (node) q3 = *reinterpret_cast<const int2*>(p + 3);
    }
};

// Codes of `cur` (yrh_internal.h).
__device__ __forceinline__ bool IsNode(int32_t code) {
    return static_cast<uint32_t>(code) < static_cast<uint32_t>(kNoRecord);
}
__device__ __forceinline__ const float4* Record(const float4* arena, int32_t code) {
    return arena + static_cast<uint32_t>(code & kUnitMask);
}
// The slot after the one `code` names, given its end-of-leaf mark.
__device__ __forceinline__ int32_t NextSlot(int32_t code, int32_t units, bool last) {
    return last ? kNoRecord : code + units;
}

__device__ __forceinline__ uint64_t LanesBelow(int lane) { return (1ull << lane) - 1ull; }

// Where this workgroup's test sums go.
__device__ __forceinline__ unsigned long long* TotalsSlot(unsigned long long* totals) {
    return totals + static_cast<int64_t>(blockIdx.x % kTotalsSlots) * kTotalsStride;
}

// Wave-level sum of the per-lane test counts (node, triangle, sphere), one
// atomic per wave and count.
__device__ __forceinline__ void AddTotals(unsigned long long* totals, uint64_t nt, uint64_t tt, uint64_t ts,
                                          int lane) {
    for (int off = 32; off > 0; off >>= 1) {
        nt += __shfl_xor(static_cast<unsigned long long>(nt), off);
        tt += __shfl_xor(static_cast<unsigned long long>(tt), off);
        ts += __shfl_xor(static_cast<unsigned long long>(ts), off);
    }
    if (lane == 0 && (nt | tt | ts) != 0) {
        unsigned long long* slot = TotalsSlot(totals);
        atomicAdd(slot, static_cast<unsigned long long>(nt));
        atomicAdd(slot + 1, static_cast<unsigned long long>(tt));
        if (ts != 0) atomicAdd(slot + 2, static_cast<unsigned long long>(ts));
    }
}

__device__ __forceinline__ void TransformRay(const float4& r0, const float4& r1, const float4& r2, float ox, float oy,
                                             float oz, float dx, float dy, float dz, float& rox, float& roy,
                                             float& roz, float& rdx, float& rdy, float& rdz) {
    // TransformPoint / TransformVector (src/core/transform.cpp:30-44), left to right.
    rox = r0.x * ox + r0.y * oy + r0.z * oz + r0.w;
    roy = r1.x * ox + r1.y * oy + r1.z * oz + r1.w;
    roz = r2.x * ox + r2.y * oy + r2.z * oz + r2.w;
    rdx = r0.x * dx + r0.y * dy + r0.z * dz;
    rdy = r1.x * dx + r1.y * dy + r1.z * dz;
    rdz = r2.x * dx + r2.y * dy + r2.z * dz;
}

// The ray-cast policy: rays from (org, dir) arrays, results to the output arrays.
template <bool kAny>
struct RayArrayPolicy {
    const TraceArgs* a;
    __device__ __forceinline__ void Begin(int32_t ray, float4& o, float4& d) const {
        o = a->org[ray];
        d = a->dir[ray];
    }
    __device__ __forceinline__ bool Finish(int32_t ray, const Best& best, int32_t inst, uint32_t nt, uint32_t tt,
                                           uint32_t ts, const float4&, const float4&, float4&, float4&) const {
        if (kAny) {
            a->occluded[ray] = best.Hit() ? 1u : 0u;
        } else {
            a->hit[ray] = best.Record();
            if (a->inst_out != nullptr) a->inst_out[ray] = best.Hit() ? inst : -1;
        }
        if (a->node_tests != nullptr) a->node_tests[ray] = nt;
        if (a->triangle_tests != nullptr) a->triangle_tests[ray] = tt;
        if (a->sphere_tests != nullptr) a->sphere_tests[ray] = ts;
        return false;
    }
};

// Rays a wave works through. The claim order is split into kParts contiguous
// stretches; workgroups are dispatched to the 8 XCDs round-robin and workgroup
// b takes part in stretch b % kParts, so each XCD works through rays that lie
// together and its L2 keeps the nodes they share.
//
// A queue with at most 64 rays per wave is dealt out by position: no atomic,
// and the rays lie on spread_waves waves (two per SIMD) if they can, so a small
// queue runs at the latency of few lanes per wave. 4096 rays on 20 k triangles,
// one context's calls one after another: 310 us at 4 rays a lane, 103, 93, 88
// and 90 us on 1, 2, 4 and 8 waves per SIMD; the short bounces of a Cornell
// frame pay for the extra waves, 2.00, 1.73, 1.73, 1.80 and 2.17 ms; 8 instanced
// cameras 48.8, 37.5, 36.0, 36.0 and 37.0 ms. A longer queue keeps a counter per
// stretch; a wave claims as many rays as it has idle lanes with one atomic and
// moves on to the next stretch when its own is used up. (Dealing the first 64 by
// position there too cost 1.29 M instanced rays 569 -> 606 us, and reading the
// counters before moving on cost 8.39 M rays 4.1 -> 4.8 ms.)
struct RaySource {
    int part;          // the stretch this wave claims from
    int parts_left;    // stretches not yet found used up (0: dealt by position)
    int32_t pos, end;  // claimed rays that no lane has yet (claim positions)
    bool drained;      // no rays left to claim
    uint32_t sum_nt, sum_tt, sum_ts;  // this lane's test counts since its last flush

    // Waves that n rays keep busy: 4 rays per lane, or spread thinner if that
    // leaves SIMDs without a wave.
    static __host__ __device__ __forceinline__ int32_t Waves(int64_t n, int32_t spread_waves) {
        const int64_t full = (n + 255) / 256, spread = n < spread_waves ? n : spread_waves;
        return static_cast<int32_t>(full > spread ? full : spread);
    }
    // False: this workgroup has nothing to do (a queue shorter than its grid
    // was sized for).
    __device__ __forceinline__ bool Init(const TraceArgs& a, int32_t n) {
        const int32_t waves_per_group = static_cast<int32_t>(blockDim.x >> 6);
        int32_t groups = (Waves(n, a.spread_waves) + waves_per_group - 1) / waves_per_group;
        if (groups > static_cast<int32_t>(gridDim.x)) groups = static_cast<int32_t>(gridDim.x);
        if (static_cast<int32_t>(blockIdx.x) >= groups) return false;
        const int32_t waves = groups * waves_per_group;
        const int32_t lanes = (n - 1) / waves + 1;
        part = static_cast<int>(blockIdx.x % kParts);
        parts_left = lanes > 64 ? kParts : 0;
        pos = end = 0;
        if (lanes <= 64) {
            const int32_t extra = groups % kParts;
            const int32_t group = part * (groups / kParts) + (part < extra ? part : extra) +
                                  static_cast<int32_t>(blockIdx.x / kParts);
            const int32_t wave = __builtin_amdgcn_readfirstlane(group * waves_per_group +
                                                                static_cast<int32_t>(threadIdx.x >> 6));
            pos = wave * lanes < n ? wave * lanes : n;
            end = pos + lanes < n ? pos + lanes : n;
        }
        drained = false;
        sum_nt = sum_tt = sum_ts = 0;
        return true;
    }
    // Claims up to `need` rays; false: none are left.
    __device__ __forceinline__ bool NextRays(const TraceArgs& a, int32_t need, int lane, int32_t n) {
        while (parts_left > 0) {
            const int32_t lo = static_cast<int32_t>(static_cast<int64_t>(part) * n / kParts);
            const int32_t hi = static_cast<int32_t>(static_cast<int64_t>(part + 1) * n / kParts);
            uint32_t base = 0;
            if (lane == 0) base = atomicAdd(a.counter + part * kPartStride, static_cast<uint32_t>(need));
            base = static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(static_cast<int>(base)));
            if (base < static_cast<uint32_t>(hi - lo)) {
                pos = lo + static_cast<int32_t>(base);
                end = hi - pos > need ? pos + need : hi;
                return true;
            }
            part = part + 1 == kParts ? 0 : part + 1;
            --parts_left;
        }
        return false;
    }
    __device__ __forceinline__ void Count(const TraceArgs& a, uint32_t nt, uint32_t tt, uint32_t ts) {
        sum_nt += nt;
        sum_tt += tt;
        sum_ts += ts;
        if (a.totals != nullptr && (sum_nt | sum_tt | sum_ts) >= 0x80000000u) {  // keep 32-bit sums from wrapping
            unsigned long long* slot = TotalsSlot(a.totals);
            atomicAdd(slot, static_cast<unsigned long long>(sum_nt));
            atomicAdd(slot + 1, static_cast<unsigned long long>(sum_tt));
            atomicAdd(slot + 2, static_cast<unsigned long long>(sum_ts));
            sum_nt = sum_tt = sum_ts = 0;
        }
    }
    // The ray index a lane without one gets, or -1.
    __device__ __forceinline__ int32_t Claim(const TraceArgs& a, int32_t ray, int lane, int32_t n) {
        uint64_t mask = Ballot(ray < 0);
        int32_t claimed = -1;
        while (mask != 0 && !drained) {
            const int32_t need = static_cast<int32_t>(__popcll(mask));
            if (pos == end && !NextRays(a, need, lane, n)) {
                drained = true;
                break;
            }
            const int32_t rank = static_cast<int32_t>(__popcll(mask & LanesBelow(lane)));
            const int32_t avail = end - pos;
            if (((mask >> lane) & 1ull) && rank < avail) claimed = pos + rank;
            pos += need < avail ? need : avail;
            mask = Ballot(ray < 0 && claimed < 0);
        }
        if (claimed >= 0 && a.order != nullptr) {
            const int32_t mapped = a.order[claimed];
            if (static_cast<uint32_t>(mapped) < static_cast<uint32_t>(n)) return mapped;
        }
        return claimed;
    }
};

__device__ __forceinline__ void ZeroNextCounters(const TraceArgs& a) {
    if (a.next_counter != nullptr && blockIdx.x == 0 && threadIdx.x < kParts) {
        a.next_counter[threadIdx.x * kPartStride] = 0u;
    }
}

// kSpheres: the tree may hold sphere slots (a scene without spheres runs the
// variant without the sphere branch, which costs its triangle tests ~2 %).
template <bool kAny, bool kSpheres, class Policy>
__device__ __forceinline__ void TraceFlatLoop(const TraceArgs& a, const Policy& pol, int2* lds_stack) {
    const int lane = static_cast<int>(threadIdx.x & 63u);
    Stack st;
    st.Init(a, lds_stack);
    ZeroNextCounters(a);
    const int32_t n = a.n_device != nullptr ? static_cast<int32_t>(*a.n_device) : a.n;
    RaySource src;
    if (!src.Init(a, n)) return;
    int32_t ray = -1;
    float dx = 0, dy = 0, dz = 0, t_min = 0;
    RayPre pre{};
    Best best = Best::None(0.0f);
    uint32_t nt = 0, tt = 0, ts = 0;
    int32_t cur = kNoRecord;  // this lane's next record

    auto start = [&](const float4& o4, const float4& d4) {
        t_min = o4.w;
        dx = d4.x; dy = d4.y; dz = d4.z;
        best = Best::None(d4.w);
        nt = 0;
        tt = 0;
        ts = 0;
        cur = kNoRecord;
        pre = Precompute(o4.x, o4.y, o4.z, dx, dy, dz);
        if (!a.empty) {
            ++nt;
            float entry;
            if (Slab(pre, a.root_lo_x, a.root_lo_y, a.root_lo_z, a.root_hi_x, a.root_hi_y, a.root_hi_z, t_min,
                     best.t, entry)) {
                cur = a.root_code;
            }
        }
    };

    while (true) {
        if (cur == kNoRecord && st.Empty() && ray >= 0) {
            src.Count(a, nt, tt, ts);
            float4 no, nd;
            if (pol.Finish(ray, best, -1, nt, tt, ts, make_float4(pre.ox, pre.oy, pre.oz, t_min),
                           make_float4(dx, dy, dz, 0.0f), no, nd)) {
                start(no, nd);
            } else {
                ray = -1;
            }
        }
        const int32_t claimed = src.Claim(a, ray, lane, n);
        if (claimed >= 0) {
            ray = claimed;
            float4 o4, d4;
            pol.Begin(ray, o4, d4);
            start(o4, d4);
        }
        // Lanes that hold a ray, or could still get one: when enough of them
        // are idle, the wave comes back here.
        const uint64_t wanted = Ballot(ray >= 0 || !src.drained);
        if (wanted == 0) break;

        while (true) {
            // A lane without a record takes its next stack entry (one beyond
            // the best hit is dropped, as the reference's pop-skip does).
            if (cur == kNoRecord && !st.Empty()) {
                int32_t code;
                float entry;
                st.Pop(code, entry);
                if (!(entry > best.t)) cur = code;
            }
            const bool node = IsNode(cur), leaf = cur < 0;
            Fetch f;
            if (cur != kNoRecord) f.Load(Record(a.arena, cur), node);
            if (node) {
                nt += 2;
                cur = InteriorStep(f.q0, f.q1, f.q2, f.q3.x, f.q3.y, pre, t_min, best.t, st);
            }
            if (leaf) {
                cur = NextSlot(cur, kSlotUnits, __float_as_int(f.q1.w) != 0);
                bool changed;
                if (kSpheres && IsSphereId(__float_as_int(f.q0.w))) {
                    ++ts;
                    changed = SphereTest(f.q0.x, f.q0.y, f.q0.z, f.q1.x, __float_as_int(f.q0.w), pre.ox, pre.oy, pre.oz,
                                         dx, dy, dz, t_min, !kAny, best);
                } else {
                    ++tt;
                    changed = TriangleTest<kAny>(f.q0, f.q1, f.q2, pre.ox, pre.oy, pre.oz, dx, dy, dz, t_min, best);
                }
                if (kAny && changed) {
                    st.Clear();
                    cur = kNoRecord;
                }
            }
            const uint64_t active = Ballot(cur != kNoRecord || !st.Empty());
            if (active == 0 || static_cast<int>(__popcll(wanted & ~active)) >= kRefillIdleLanes) break;
        }
    }
    if (a.totals != nullptr) AddTotals(a.totals, src.sum_nt, src.sum_tt, src.sum_ts, lane);
}

template <bool kAny, bool kSpheres, class Policy>
__device__ __forceinline__ void TraceTwoLevelLoop(const TraceArgs& a, const Policy& pol, int2* lds_stack) {
    const int lane = static_cast<int>(threadIdx.x & 63u);
    Stack st;
    st.Init(a, lds_stack);
    ZeroNextCounters(a);
    const int32_t n = a.n_device != nullptr ? static_cast<int32_t>(*a.n_device) : a.n;
    RaySource src;
    if (!src.Init(a, n)) return;
    int32_t ray = -1;
    float ox = 0, oy = 0, oz = 0, dx = 0, dy = 0, dz = 0, t_min = 0;  // the world ray
    // The ray being traversed: the world ray in the TLAS, the object ray inside
    // a BLAS (the world ray's reciprocals are recomputed, bit-identically, when
    // the BLAS is left), so one set of registers serves both levels. tdx..tdz:
    // its direction.
    RayPre pre{};
    float tdx = 0, tdy = 0, tdz = 0;
    Best best = Best::None(0.0f);
    int32_t best_inst = -1;
    uint32_t nt = 0, tt = 0, ts = 0;
    // The BLAS being traversed: its hit, and the stack level below it.
    bool in_blas = false;
    uint32_t blas_base = 0;
    int32_t cur_inst = -1;
    Best bbest = Best::None(0.0f);
    int32_t cur = kNoRecord;   // this lane's next record
    int32_t inst = kNoRecord;  // the next instance slot of the TLAS leaf being expanded

    auto start = [&](const float4& o4, const float4& d4) {
        ox = o4.x; oy = o4.y; oz = o4.z; t_min = o4.w;
        dx = d4.x; dy = d4.y; dz = d4.z;
        best = Best::None(d4.w);
        best_inst = -1;
        nt = 0;
        tt = 0;
        ts = 0;
        in_blas = false;
        inst = cur = kNoRecord;
        pre = Precompute(ox, oy, oz, dx, dy, dz);
        if (!a.empty) {
            ++nt;
            float entry;
            if (Slab(pre, a.root_lo_x, a.root_lo_y, a.root_lo_z, a.root_hi_x, a.root_hi_y, a.root_hi_z, t_min,
                     best.t, entry)) {
                if (a.root_code < 0) {
                    inst = a.root_code;
                } else {
                    cur = a.root_code;
                }
            }
        }
    };

    while (true) {
        const bool busy = in_blas || inst != kNoRecord || cur != kNoRecord || !st.Empty();
        if (!busy && ray >= 0) {
            src.Count(a, nt, tt, ts);
            float4 no, nd;
            if (pol.Finish(ray, best, best_inst, nt, tt, ts, make_float4(ox, oy, oz, t_min),
                           make_float4(dx, dy, dz, 0.0f), no, nd)) {
                start(no, nd);
            } else {
                ray = -1;
            }
        }
        const int32_t claimed = src.Claim(a, ray, lane, n);
        if (claimed >= 0) {
            ray = claimed;
            float4 o4, d4;
            pol.Begin(ray, o4, d4);
            start(o4, d4);
        }
        const uint64_t wanted = Ballot(ray >= 0 || !src.drained);
        if (wanted == 0) break;

        while (true) {
            // One record per iteration, as in the flat loop: a BLAS leaf's
            // triangles one by one, or a node. A lane that finishes a BLAS or
            // pops a TLAS leaf tries its next instance in the same iteration,
            // and an instance whose root box is hit goes straight to its root
            // record (no stack round trip): fewer iterations per instance
            // visit, the same operations in the same order.
            if (cur == kNoRecord) {
                if (in_blas && st.sp == blas_base) {
                    // BLAS finished: accept only a strictly closer hit (two_level_bvh.cpp:474);
                    // an occlusion query accepts any hit within [t_min, t_max].
                    if (bbest.Hit() && (kAny || bbest.t < best.t)) {
                        best = bbest;
                        best_inst = cur_inst;
                        if (kAny) {
                            st.Clear();
                            inst = kNoRecord;
                        }
                    }
                    in_blas = false;
                    pre = Precompute(ox, oy, oz, dx, dy, dz);
                } else if ((in_blas || inst == kNoRecord) && !st.Empty()) {
                    int32_t code;
                    float entry;
                    st.Pop(code, entry);
                    const float bound = in_blas ? bbest.t : best.t;
                    if (!(entry > bound)) {
                        if (!in_blas && code < 0) {
                            inst = code;
                        } else {
                            cur = code;
                        }
                    }
                }
                if (!in_blas && inst != kNoRecord && cur == kNoRecord) {
                    const DevInstanceSlot m = *reinterpret_cast<const DevInstanceSlot*>(Record(a.arena, inst));
                    const int32_t slot_id = __float_as_int(m.hi.w);
                    const int32_t root = __float_as_int(m.lo.w);
                    inst = NextSlot(inst, kInstanceUnits, (root & kLastInstanceBit) != 0);
                    if (kSpheres && IsSphereId(slot_id)) {
                        // A TLAS sphere (IntersectTlasSphere, two_level_bvh.cpp:231-253):
                        // tested against the world ray, no instance.
                        ++ts;
                        if (SphereTest(m.r0.x, m.r0.y, m.r0.z, m.r0.w, slot_id, ox, oy, oz, dx, dy, dz, t_min, !kAny,
                                       best)) {
                            best_inst = -1;
                            if (kAny) {
                                st.Clear();
                                inst = kNoRecord;
                            }
                        }
                    } else {
                        // Object ray, BLAS root box.
                        cur_inst = slot_id;
                        float bx, by, bz;
                        TransformRay(m.r0, m.r1, m.r2, ox, oy, oz, dx, dy, dz, bx, by, bz, tdx, tdy, tdz);
                        const RayPre bpre = Precompute(bx, by, bz, tdx, tdy, tdz);
                        ++nt;
                        float entry;
                        if (Slab(bpre, m.lo.x, m.lo.y, m.lo.z, m.hi.x, m.hi.y, m.hi.z, t_min, best.t, entry)) {
                            // The root's entry distance is within [t_min, best t], so the
                            // stack pop it replaces would always have taken it.
                            pre = bpre;
                            bbest = Best::None(best.t);
                            blas_base = st.sp;
                            in_blas = true;
                            cur = root & ~kLastInstanceBit;
                        }
                    }
                }
            }
            const bool node = IsNode(cur), leaf = cur < 0;
            Fetch f;
            if (cur != kNoRecord) f.Load(Record(a.arena, cur), node);
            if (node) {
                nt += 2;
                cur = InteriorStep(f.q0, f.q1, f.q2, f.q3.x, f.q3.y, pre, t_min, in_blas ? bbest.t : best.t, st);
                if (cur < 0 && !in_blas) {  // a TLAS leaf: its instances come next
                    inst = cur;
                    cur = kNoRecord;
                }
            }
            if (leaf) {
                ++tt;
                cur = NextSlot(cur, kSlotUnits, __float_as_int(f.q1.w) != 0);
                if (TriangleTest<kAny>(f.q0, f.q1, f.q2, pre.ox, pre.oy, pre.oz, tdx, tdy, tdz, t_min, bbest) && kAny) {
                    cur = kNoRecord;
                    st.sp = blas_base;  // finish this BLAS now
                }
            }
            const uint64_t active = Ballot(in_blas || inst != kNoRecord || cur != kNoRecord || !st.Empty());
            if (active == 0 || static_cast<int>(__popcll(wanted & ~active)) >= kRefillIdleLanes) break;
        }
    }
    if (a.totals != nullptr) AddTotals(a.totals, src.sum_nt, src.sum_tt, src.sum_ts, lane);
}

}  // namespace trav

// Fills the launch arguments (grid, stack spill region, counters) of one
// traversal over `r`'s queue (yrh_trace.hip).
int PrepareTraceArgs(yrh_context* ctx, const TraceRequest& r, trav::TraceArgs& a, int& grid, int& block);
// Dynamic LDS bytes of a traversal launch with `block` threads.
size_t LdsBytes(const trav::TraceArgs& a, int block);

}  // namespace yrh
