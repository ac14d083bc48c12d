"""Render passes with a bounce's shadow rays on a second stream, one or two
bounces behind the path segments, leave the same film and counters as the
one-stream sequence: every per-path operation keeps its order, so the FP64
films are compared byte for byte. Each setting has a context of its own: what
a context has allocated before must not decide what is compared."""
import contextlib

import numpy as np
import pytest
import torch

from yaoray_amd import Device, Scene
from yaoray_amd import native as N
from yaoray_amd.api import YrhError

pytestmark = pytest.mark.gpu

MIB = 1 << 20


@contextlib.contextmanager
def context(overlap):
    dev = Device(0)
    try:
        dev.set_render_overlap(overlap)
        yield dev
        dev.synchronize()
    finally:
        dev.close()


def both(run):
    out = []
    for overlap in (False, True):
        with context(overlap) as dev:
            out.append(run(dev))
    return out


def instanced():
    # glass instances: transparent shadow walks; sky + sun environment
    s = Scene.instanced(instances=150, subdivisions=2, variants=6, env_width=64, env_height=32, seed=4)
    s.build_accel()
    return s


@pytest.mark.parametrize("scene", ["cornell", "instanced"])
def test_overlapped_bounces_match_sequential(scene):
    if scene == "cornell":
        s = Scene.cornell(1)
        s.build_accel()
        w, h, spp, depth, batch = 96, 64, 16, 8, 8
    else:
        s = instanced()
        w, h, spp, depth, batch = 96, 64, 8, 12, 4
    (f0, st0), (f1, st1) = both(lambda dev: dev.render(s, w, h, spp, max_depth=depth, batch=batch, seed=3))
    assert f1.tobytes() == f0.tobytes()
    assert st1 == st0
    assert f0["samples"].sum() == w * h * spp


@pytest.mark.parametrize("graph", [False, True])
def test_overlapped_batches_match_sequential(graph):
    s = instanced()
    jobs = [s.render_desc(w, h, spp) for w, h, spp in ((64, 48, 6), (37, 29, 9), (96, 17, 4))]

    def run(dev):
        dev.upload_scene(s)
        dev.upload_shading(s)
        films, _, passes, stats = dev.render_batch(jobs, max_depth=10, paths_per_pass=5000, use_graph=graph)
        assert passes > 3
        return b"".join(f.tobytes() for f in films), stats

    (f0, st0), (f1, st1) = both(run)
    assert f1 == f0
    assert st1 == st0


def guided(dev, s):
    dev.guide_configure([-0.1, -0.1, -0.1], [10.1, 4.1, 10.1], log2_table_size=16, min_resolution=8,
                        max_resolution=128, learning_rate=3e-3, guide_fraction=0.5, sample_capacity=1 << 16, seed=7)
    dev.upload_scene(s)
    dev.upload_shading(s)


def room():
    s = Scene.room(furniture_triangles=20000, env_width=64, env_height=32)
    s.build_accel()
    return s


def test_overlapped_recording_matches_sequential():
    """The records hold the radiance so far, so they show a Resolve that comes too
    early or late."""
    s = room()

    def run(dev):
        guided(dev, s)
        dev.guide_set_mode(N.GUIDE_RECORD)
        film, stats = dev.render(s, 64, 36, 4, max_depth=6, upload=False, batch=4, seed=9)
        samples = dev.guide_read_samples(1 << 16)
        return film.tobytes(), stats, samples[np.lexsort(samples.T)]

    (f0, st0, s0), (f1, st1, s1) = both(run)
    assert f1 == f0
    assert st1 == st0
    assert len(s0) > 10000 and s1.tobytes() == s0.tobytes()


def test_overlapped_guided_bounces_match_sequential():
    s = room()
    with context(True) as dev:
        guided(dev, s)
        dev.guide_set_mode(N.GUIDE_RECORD)
        dev.render(s, 64, 36, 2, max_depth=6, upload=False, seed=9)
        dev.guide_train(4, 4096)
        params = dev.guide_params()

    def run(dev):
        guided(dev, s)
        dev.guide_set_params(*params)
        dev.guide_set_mode(N.GUIDE_SAMPLE)
        return dev.render(s, 64, 36, 8, max_depth=6, upload=False, batch=8, seed=11)[0]

    f0, f1 = both(run)
    assert f1.tobytes() == f0.tobytes()


PATHS = 512 * 256 * 8  # of the passes below
QUEUE = 80 * PATHS     # a shadow queue of one entry per path


def taken(dev, s):
    """Device memory that a pass of PATHS paths takes on top of what the context has."""
    before = torch.cuda.mem_get_info()[0]
    dev.render(s, 512, 256, 8, max_depth=3, upload=False, batch=8)
    return before - torch.cuda.mem_get_info()[0]


def test_second_shadow_queue_follows_the_overlap_setting():
    """The two-bounce lag needs a second shadow queue. A context whose first pass
    ran on one stream gets it when overlap comes on."""
    s = Scene.cornell(1)
    s.build_accel()
    with context(True) as dev:
        dev.upload_scene(s)
        dev.upload_shading(s)
        whole = taken(dev, s)
    with context(False) as dev:
        dev.upload_scene(s)
        dev.upload_shading(s)
        alone = taken(dev, s)
        assert whole - alone > 0.9 * QUEUE
        dev.set_render_overlap(True)
        assert taken(dev, s) > 0.9 * QUEUE
        assert taken(dev, s) < 0.1 * QUEUE


def test_recording_passes_take_no_second_shadow_queue():
    """They wait for the Resolve of the bounce before and need the memory for
    their records; a sampling pass of the same size then takes it."""
    s = room()
    with context(True) as dev:
        guided(dev, s)
        dev.guide_set_cell_budget(0)
        dev.guide_set_mode(N.GUIDE_RECORD)
        taken(dev, s)
        dev.guide_set_mode(N.GUIDE_SAMPLE)
        assert taken(dev, s) > 0.9 * QUEUE


def test_second_shadow_queue_is_given_back_when_memory_is_short():
    s = Scene.cornell(1)
    s.build_accel()
    with context(True) as dev:
        dev.upload_scene(s)
        dev.upload_shading(s)
        taken(dev, s)
        f0 = dev.film_read(512, 256)
        before, total = torch.cuda.mem_get_info()
        with pytest.raises(YrhError, match="out of memory"):
            dev.alloc(2 * total)
        assert torch.cuda.mem_get_info()[0] - before > 0.9 * QUEUE
        assert taken(dev, s) > 0.9 * QUEUE
        assert dev.film_read(512, 256).tobytes() == f0.tobytes()


@pytest.mark.parametrize("overlap", [False, True])
def test_suggested_pass_counts_what_the_context_holds(overlap):
    """Half of (free memory + held path state) over the bytes of a path; with a
    proposal and this depth below the cap, so the held bytes can be told."""
    s, depth = Scene.cornell(1), 1000
    s.build_accel()
    with context(overlap) as dev:
        guided(dev, s)
        free = torch.cuda.mem_get_info()[0]
        per_path = free / 2 / dev.suggest_paths_per_pass(depth)
        grown = taken(dev, s)
        assert grown > 0.9 * QUEUE
        held = dev.suggest_paths_per_pass(depth) * 2 * per_path - torch.cuda.mem_get_info()[0]
        assert 0.5 * grown < held < grown + 4 * per_path + 16 * MIB


@pytest.mark.parametrize("overlap", [False, True])
def test_passes_in_a_callers_graph(overlap):
    """A pass that a caller captures after an eager one allocates nothing, each
    replay adds what an eager pass adds, and the graph does not use the second
    shadow queue, which the context may give back."""
    s = Scene.cornell(1)
    s.build_accel()
    with context(True) as dev:
        dev.upload_scene(s)
        dev.upload_shading(s)
        desc = s.render_desc(64, 48, 4, 5)
        desc.sample_count = 4
        dev.film_reset(64, 48)
        for _ in range(4):
            dev.render_pass(desc)
        dev.synchronize()
        eager = dev.film_read(64, 48).tobytes()
        dev.set_render_overlap(overlap)
        stream = torch.cuda.ExternalStream(dev._lib.yrh_stream(dev._ctx))
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=stream, capture_error_mode="thread_local"):
            dev.render_pass(desc)
        for turn in range(3):
            if turn == 1:
                with pytest.raises(YrhError, match="out of memory"):
                    dev.alloc(2 * torch.cuda.mem_get_info()[1])
                reuse = torch.full((16 * MIB,), 7, dtype=torch.uint8, device="cuda")
                torch.cuda.synchronize()
            dev.film_reset(64, 48)
            for k in range(4):
                if k == 2 and turn == 2:
                    dev.render_pass(desc)
                else:
                    with torch.cuda.stream(stream):
                        graph.replay()
            dev.synchronize()
            assert dev.film_read(64, 48).tobytes() == eager, turn
            assert turn == 0 or bool((reuse == 7).all())
