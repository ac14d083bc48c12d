"""Large copies to the host go through pinned buffers on several threads: every byte
arrives, in both directions, at sizes around the chunk and thread limits."""
import numpy as np
import pytest

from yaoray_amd import Device
from yaoray_amd.api import DeviceBuffer

pytestmark = pytest.mark.gpu

MIB = 1 << 20


# Staged from 6 MiB on, 1 MiB a chunk, a thread per two chunks up to eight.
@pytest.mark.parametrize("nbytes", [6 * MIB - 1, 6 * MIB, 6 * MIB + 1, 7 * MIB + 4093, 9 * MIB + 1, 12 * MIB, 15 * MIB + 1,
                                    16 * MIB, 17 * MIB + 1, 32 * MIB, 41 * MIB + 7])
@pytest.mark.parametrize("first", [True, False])
def test_large_copies_arrive_whole(nbytes, first):
    """As a context's first large copy (plain under 32 MiB) and after one."""
    rng = np.random.default_rng(nbytes)
    dev = Device(0)
    try:
        if not first:
            DeviceBuffer(dev, 32 * MIB).download(np.uint8, 32 * MIB)
        buf = DeviceBuffer(dev, nbytes + 64)
        guard = np.full(64, 7, np.uint8)
        for _ in range(1 if first else 3):
            a = rng.integers(0, 256, nbytes, np.uint8)
            buf.upload(np.concatenate([np.zeros(nbytes, np.uint8), guard]))
            buf.upload(a)
            out = np.full(nbytes + 64, 3, np.uint8)
            dev._check(dev._lib.yrh_copy_to_host(dev._ctx, out.ctypes.data, buf.ptr, nbytes), "copy_to_host")
            assert np.array_equal(out[:nbytes], a)
            assert (out[nbytes:] == 3).all()
            assert np.array_equal(buf.download(np.uint8, nbytes + 64)[nbytes:], guard)
        buf.free()
    finally:
        dev.close()


@pytest.mark.parametrize("mib", [8, 16])
def test_uploads_cost_no_more_than_a_plain_copy(mib):
    """Scene arrays of some MiB to the device, against torch's copy of the same
    pageable memory (through the context's pinned buffers they took 1.3 to 1.4
    times as long)."""
    import time

    import torch
    a = np.ones(mib * MIB, np.uint8)
    t, on_device = torch.from_numpy(a), torch.empty(a.nbytes, dtype=torch.uint8, device="cuda")
    dev = Device(0)
    try:
        buf = DeviceBuffer(dev, a.nbytes)
        ours, plain = [], []
        for _ in range(30):
            t0 = time.perf_counter()
            buf.upload(a)
            t1 = time.perf_counter()
            on_device.copy_(t)
            torch.cuda.synchronize()
            ours.append(t1 - t0)
            plain.append(time.perf_counter() - t1)
        buf.free()
    finally:
        dev.close()
    assert np.percentile(ours, 25) < 1.15 * np.percentile(plain, 25)


def test_destinations_that_are_not_pageable(device):
    """Pinned memory takes the copy directly (through the context's buffers it
    took 1.8 times as long), device memory too."""
    import time

    import torch
    n = 64 * MIB
    a = np.random.default_rng(3).integers(0, 256, n, np.uint8)
    buf = DeviceBuffer(device, n).upload(a)
    pinned, on_device = torch.zeros(n, dtype=torch.uint8, pin_memory=True), torch.zeros(n, dtype=torch.uint8, device="cuda")
    torch.cuda.synchronize()
    ours, plain = [], []
    for _ in range(12):
        t0 = time.perf_counter()
        device._check(device._lib.yrh_copy_to_host(device._ctx, pinned.data_ptr(), buf.ptr, n), "copy_to_host")
        ours.append(time.perf_counter() - t0)
    assert np.array_equal(pinned.numpy(), a)
    device._check(device._lib.yrh_copy_to_host(device._ctx, on_device.data_ptr(), buf.ptr, n), "copy_to_host")
    assert np.array_equal(on_device.cpu().numpy(), a)
    for _ in range(12):
        t0 = time.perf_counter()
        pinned.copy_(on_device)
        torch.cuda.synchronize()
        plain.append(time.perf_counter() - t0)
    buf.free()
    assert np.percentile(ours, 25) < 1.3 * np.percentile(plain, 25)
