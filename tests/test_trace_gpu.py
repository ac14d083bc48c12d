"""GPU parity of the HIP traversal kernels against the CPU oracle, through the C ABI.

Bar: bit-exact hit ids, t, barycentrics and node/triangle counters (integer and
index work on identical FP32 arithmetic), occlusion == closest hit found.
"""
import numpy as np
import pytest

from oracle import oracle_py as O
from tests.helpers import MeshArrays, rays, same_bits, trs
from yaoray_amd import Scene, random_rays

pytestmark = pytest.mark.gpu


def gpu_closest(device, scene, org, d):
    device.upload_scene(scene)
    return device.trace_closest(org, d, counters=True)


def assert_same(g, o, keys=("t", "u", "v", "triangle", "node_tests", "triangle_tests")):
    for k in keys:
        if not same_bits(g[k], o[k]):
            bad = np.nonzero(g[k].view(np.uint32) != o[k].view(np.uint32))[0] if g[k].dtype == np.float32 else \
                np.nonzero(g[k] != o[k])[0]
            raise AssertionError(f"{k}: {len(bad)} mismatches, first at {bad[:5]}: gpu {g[k][bad[:5]]} "
                                 f"oracle {o[k][bad[:5]]}")


@pytest.fixture(scope="module")
def tri_scene():
    s = Scene.triangles(60000, seed=2)
    s.build_accel()
    return s


def workload_rays(scene, n_random=40000, res=160):
    o1, d1 = scene.camera_rays(res, res)
    o2, d2 = random_rays(n_random, seed=3)
    return np.concatenate([o1, o2]), np.concatenate([d1, d2])


def test_flat_closest_matches_oracle(device, tri_scene):
    org, d = workload_rays(tri_scene)
    g = gpu_closest(device, tri_scene, org, d)
    v, i, p = tri_scene.geometry()
    o = O.trace_flat(v, i, p, tri_scene.flat_bvh(), org, d)
    assert_same(g, o)
    assert np.all(g["instance"] == -1)
    assert 0.2 < (g["triangle"] >= 0).mean() < 1.0


def test_flat_any_matches_oracle(device, tri_scene):
    org, d = workload_rays(tri_scene, n_random=20000, res=100)
    device.upload_scene(tri_scene)
    g = device.trace_any(org, d, counters=True)
    v, i, p = tri_scene.geometry()
    o = O.trace_flat(v, i, p, tri_scene.flat_bvh(), org, d, occlusion=True)
    c = O.trace_flat(v, i, p, tri_scene.flat_bvh(), org, d)
    assert np.array_equal(g["occluded"], o["occluded"])
    assert np.array_equal(g["occluded"].astype(bool), c["triangle"] >= 0)
    assert_same(g, o, keys=("node_tests", "triangle_tests"))


def test_finite_segments_and_tmin(device, tri_scene):
    org, d = random_rays(20000, seed=21)
    rng = np.random.default_rng(4)
    d[:, 3] = rng.uniform(0.0, 0.5, len(d)).astype(np.float32)
    org[:, 3] = rng.uniform(0.0, 0.05, len(d)).astype(np.float32)
    g = gpu_closest(device, tri_scene, org, d)
    v, i, p = tri_scene.geometry()
    o = O.trace_flat(v, i, p, tri_scene.flat_bvh(), org, d)
    assert_same(g, o)
    ga = device.trace_any(org, d)
    assert np.array_equal(ga["occluded"].astype(bool), o["triangle"] >= 0)


def test_axis_parallel_and_degenerate_rays(device):
    # Rays with zero direction components (1/d = +-inf, 0*inf = NaN on slab planes),
    # rays lying exactly on box faces, and a zero-length direction.
    m = MeshArrays()
    grid = []
    for x in range(6):
        for y in range(6):
            grid.append([[x, y, 0], [x + 1, y, 0], [x, y + 1, 0]])
            grid.append([[x, y, 1], [x + 1, y, 1], [x, y + 1, 1]])
    m.add_triangles(np.array(grid, np.float32))
    s = m.scene()
    s.build_accel()
    origins, dirs = [], []
    for x in np.linspace(-0.5, 6.5, 15):
        for y in np.linspace(-0.5, 6.5, 15):
            origins += [(x, y, 2.0), (x, y, -1.0), (x, y, 0.0), (x, -1.0, 0.5)]
            dirs += [(0, 0, -1), (0, 0, 1), (1, 0, 0), (0, 1, 0)]
    origins += [(0.2, 0.2, 2.0), (0.0, 0.0, 0.0), (1.0, 1.0, 1.0)]
    dirs += [(0, 0, 0), (-0.0, 0.0, -1.0), (0.0, -0.0, -1.0)]
    org, d = rays(origins, dirs)
    g = gpu_closest(device, s, org, d)
    v, i, p = s.geometry()
    o = O.trace_flat(v, i, p, s.flat_bvh(), org, d)
    assert_same(g, o)


def test_empty_scene_and_single_triangle(device):
    empty = MeshArrays().scene()
    empty.build_accel()
    org, d = rays([(0, 0, 1)] * 3, [(0, 0, -1)] * 3)
    g = gpu_closest(device, empty, org, d)
    assert np.all(g["triangle"] == -1) and np.all(g["node_tests"] == 0)
    assert np.all(g["t"] == np.inf)
    one = MeshArrays().add_test_triangle(0.0).scene()
    one.build_accel()
    g = gpu_closest(device, one, org, d)
    assert np.all(g["triangle"] == 0) and np.all(np.abs(g["t"] - 1.0) < 1e-6)
    assert np.all(g["triangle_tests"] == 1)


def test_deep_tree_uses_stack_spill(device):
    # Triangles at x = 4^k make the SAH peel about one triangle per level, so
    # the tree is deeper than the 16 LDS stack levels; rays travelling along +x
    # in the triangles' plane hit both children at every level and fill the
    # stack to the tree depth.
    tris = []
    for k in range(59):
        x = 4.0 ** k
        tris.append([[x, 0, 0], [x * 1.05, 0, 0], [x, 0.5 * max(1.0, x * 0.01), 0]])
    m = MeshArrays().add_triangles(np.array(tris, np.float32))
    s = m.scene()
    s.build_accel()
    assert s.flat_bvh().max_depth > 20
    xs = np.array([4.0 ** k * 1.01 for k in range(59)] * 4, np.float32)
    ys = np.repeat([0.05, 0.1, 0.2, 0.45], 59).astype(np.float32)
    origins = np.stack([xs, ys, np.full_like(xs, 1.0)], 1)
    org, d = rays(origins, [(0, 0, -1)] * len(xs))
    o2, d2 = rays([(-1.0, 0.1, 0.0)] * 4, [(1, 0, 0), (1, 0.001, 0), (1, 0, 0.001), (1, 0.01, 0)])
    org, d = np.concatenate([org, o2]), np.concatenate([d, d2])
    g = gpu_closest(device, s, org, d)
    v, i, p = s.geometry()
    o = O.trace_flat(v, i, p, s.flat_bvh(), org, d)
    assert_same(g, o)


def overlapping_tree(bvh, counts):
    """A root over two leaves of `counts` primitives that share some, some
    positions of primitive_indices in neither; box = the given tree's root box."""
    from yaoray_amd.api import BvhArrays
    n = len(bvh.primitive_indices)
    nodes = np.repeat(bvh.nodes[:1], 3)
    nodes["payload_offset"], nodes["primitive_count"] = [2, 2, n - counts[1]], [0, counts[0], counts[1]]
    assert 2 + counts[0] > n - counts[1]  # they overlap
    return BvhArrays(nodes, bvh.primitive_indices, bvh.primitives, 2)


@pytest.mark.parametrize("kind", ["flat", "two_level"])
def test_leaves_that_share_primitives(device, kind):
    """Leaves longer than 15 primitives, overlapping ranges, primitives of no
    leaf: the device's per-leaf slots hold what each leaf names."""
    org, d = random_rays(3000, seed=12)
    if kind == "flat":
        s = Scene.triangles(300, seed=3)
        s.build_accel()
        v, i, p = s.geometry()
        t = overlapping_tree(s.flat_bvh(), (200, 120))
        g = s.geometry_desc()
        g.flat = t.desc()
        o = O.trace_flat(v, i, p, t, org, d)
    else:
        s = Scene.instanced(instances=20, subdivisions=2, variants=3, env_width=8, env_height=4, seed=6)
        s.build_accel()
        v, i, p = s.geometry()
        tl, tp, inst = s.tlas()
        org[:, :3] = org[:, :3] * (40.0, 6.0, 40.0) - (20.0, 1.0, 20.0)
        t = overlapping_tree(tl, (13, 9))
        g = s.geometry_desc()
        flat = t.desc()
        flat.primitives, flat.primitive_count = None, 0
        g.tlas = flat
        o = O.trace_two_level(v, i, p, [s.blas(k) for k in range(s.info.blas_count)], inst, t, tp, org, d)
    device.upload_geometry(g)
    r = device.trace_closest(org, d, counters=True)
    assert_same(r, o)
    assert kind == "flat" or same_bits(r["instance"], o["instance"])
    assert (r["triangle"] >= 0).any()


def test_leaves_that_name_the_same_range_share_slots(device):
    """512 leaves over the same 1000 primitives: their slots are held once (25 MB
    otherwise), and every leaf finds them."""
    import torch

    from yaoray_amd.api import BvhArrays
    s = Scene.triangles(1000, seed=3)
    s.build_accel()
    v, i, p = s.geometry()
    b = s.flat_bvh()
    nodes = []

    def add(levels):
        nodes.append(b.nodes[0].copy())
        k = len(nodes) - 1
        if levels == 0:
            nodes[k]["payload_offset"], nodes[k]["primitive_count"] = 0, len(b.primitive_indices)
            return
        add(levels - 1)
        nodes[k]["payload_offset"], nodes[k]["primitive_count"] = len(nodes), 0
        add(levels - 1)

    add(9)
    t = BvhArrays(np.array(nodes), b.primitive_indices, b.primitives, 10)
    g = s.geometry_desc()
    device.upload_geometry(g)
    device.synchronize()
    before = torch.cuda.mem_get_info()[0]
    g.flat = t.desc()
    device.upload_geometry(g)
    assert before - torch.cuda.mem_get_info()[0] < 8 << 20
    org, d = random_rays(64, seed=12)
    assert_same(device.trace_closest(org, d, counters=True), O.trace_flat(v, i, p, t, org, d))


def test_upload_time_is_linear_in_the_number_of_meshes(device):
    """6000 meshes of 100 triangles, 0.06 s (2.7 s where each mesh moves all those
    before it; 12000 meshes took 40 s)."""
    import time

    from yaoray_amd.api import PRIMITIVE_DTYPE, VERTEX_DTYPE
    meshes, tris = 6000, 100
    rng = np.random.default_rng(2)
    v = np.zeros(meshes * tris * 3, VERTEX_DTYPE)
    v["position"] = (rng.uniform(-1, 1, (meshes * tris, 1, 3)) + rng.uniform(-0.1, 0.1, (meshes * tris, 3, 3))).reshape(-1, 3)
    p = np.zeros(meshes, PRIMITIVE_DTYPE)
    p["first_index"], p["index_count"] = np.arange(meshes) * 3 * tris, 3 * tris
    s = Scene.from_arrays(v, np.arange(len(v), dtype=np.uint32), p, np.arange(meshes, dtype=np.int32),
                          np.stack([trs((0, 0, 0), (0, 1, 0), 0, 1.0)] * meshes))
    s.build_accel()
    assert s.info.blas_count == 6000
    t = time.perf_counter()
    device.upload_scene(s)
    assert time.perf_counter() - t < 1.0


@pytest.mark.parametrize("kind", ["flat", "two_level"])
def test_hits_on_triangles_without_a_flat_index(device, kind):
    """A caller's tree may hold triangles whose flat index is -1: they shorten
    the ray and occlude as any other, and their hit reports id -1."""
    import ctypes as C

    from yaoray_amd import native as N
    org, d = random_rays(20000, seed=31)
    if kind == "flat":
        s = Scene.triangles(3000, seed=3)
        trees = lambda: [s.flat_bvh()]  # noqa: E731
    else:
        s = Scene.instanced(instances=60, subdivisions=2, variants=3, env_width=8, env_height=4, seed=6)
        org[:, :3] = org[:, :3] * (40.0, 6.0, 40.0) - (20.0, 1.0, 20.0)
        trees = lambda: [s.blas(k) for k in range(s.info.blas_count)]  # noqa: E731
    s.build_accel()
    v, i, p = s.geometry()
    g, trees = s.geometry_desc(), trees()
    for t in trees:
        t.primitives["flat_triangle_index"][::2] = -1
    if kind == "flat":
        g.flat = trees[0].desc()
        oracle = lambda **k: O.trace_flat(v, i, p, trees[0], org, d, **k)  # noqa: E731
    else:
        blases = (N.BvhDesc * len(trees))(*[t.desc() for t in trees])
        g.blases = C.cast(blases, C.c_void_p)
        tl, tp, inst = s.tlas()
        oracle = lambda **k: O.trace_two_level(v, i, p, trees, inst, tl, tp, org, d, **k)  # noqa: E731
    device.upload_geometry(g)
    r, o = device.trace_closest(org, d, counters=True), oracle()
    assert_same(r, o)
    assert kind == "flat" or same_bits(r["instance"], o["instance"])
    hidden = np.isfinite(r["t"]) & (r["triangle"] == -1)
    assert 0.005 < hidden.mean() and (r["triangle"] >= 0).any()
    a, o = device.trace_any(org, d, counters=True), oracle(occlusion=True)
    assert np.array_equal(a["occluded"], o["occluded"]) and (a["occluded"][hidden] == 1).all()
    assert_same(a, o, keys=("node_tests", "triangle_tests"))


def test_launch_shape_invariance(device, tri_scene):
    org, d = workload_rays(tri_scene, n_random=30000, res=64)
    base = gpu_closest(device, tri_scene, org, d)
    try:
        for bpc, bs in ((1, 64), (2, 128), (8, 256)):
            device.set_trace_config(bpc, bs)
            assert_same(device.trace_closest(org, d, counters=True), base)
    finally:
        device.set_trace_config(4, 256)


def two_level_scene():
    s = Scene.instanced(instances=500, subdivisions=3, variants=4, env_width=8, env_height=4, seed=4)
    s.build_accel()
    return s


@pytest.mark.parametrize("shape", [(4, 256), (1, 64), (3, 128)])
@pytest.mark.parametrize("n", [1, 5, 63, 2047, 2049, 16385, 131072, 131073, 150001])
def test_every_ray_is_claimed_once(device, n, shape):
    """Queue lengths around the sizes where rays are dealt by position, spread
    over more waves than they fill, or claimed from the range counters."""
    s = Scene.triangles(300, seed=3)
    s.build_accel()
    org, d = random_rays(n, seed=21)
    v, i, p = s.geometry()
    o = O.trace_flat(v, i, p, s.flat_bvh(), org, d)
    device.upload_scene(s)
    device.set_trace_config(*shape)
    try:
        assert_same(device.trace_closest(org, d, counters=True), o)
        g = device.trace_any(org, d)
    finally:
        device.set_trace_config(4, 256)
    assert np.array_equal(g["occluded"].astype(bool), o["triangle"] >= 0)


def test_two_level_closest_and_any_match_oracle(device):
    s = two_level_scene()
    v, i, p = s.geometry()
    tl, tp, inst = s.tlas()
    blases = [s.blas(k) for k in range(s.info.blas_count)]
    o1, d1 = s.camera_rays(240, 135)
    rng = np.random.default_rng(5)
    o2 = np.zeros((20000, 4), np.float32)
    o2[:, :3] = rng.uniform([-30, 0, -30], [30, 5, 30], (20000, 3))
    o2[:, 3] = 1e-5
    dd = rng.normal(size=(20000, 3))
    d2 = np.zeros((20000, 4), np.float32)
    d2[:, :3] = dd / np.linalg.norm(dd, axis=1, keepdims=True)
    d2[:, 3] = np.inf
    org, d = np.concatenate([o1, o2]), np.concatenate([d1, d2])
    g = gpu_closest(device, s, org, d)
    o = O.trace_two_level(v, i, p, blases, inst, tl, tp, org, d)
    assert_same(g, o, keys=("t", "u", "v", "triangle", "instance", "node_tests", "triangle_tests"))
    ga = device.trace_any(org, d, counters=True)
    oa = O.trace_two_level(v, i, p, blases, inst, tl, tp, org, d, occlusion=True)
    assert np.array_equal(ga["occluded"], oa["occluded"])
    assert np.array_equal(ga["occluded"].astype(bool), o["triangle"] >= 0)
    assert_same(ga, oa, keys=("node_tests", "triangle_tests"))


def test_two_level_scaled_rotated_instances(device):
    m = MeshArrays()
    rng = np.random.default_rng(8)
    c = rng.uniform(-1, 1, (300, 1, 3))
    m.add_triangles(c + rng.uniform(-0.1, 0.1, (300, 3, 3)))
    mats = [trs(rng.uniform(-4, 4, 3), rng.normal(size=3), rng.uniform(0, 360), rng.uniform(0.2, 2.0))
            for _ in range(64)]
    s = m.scene(np.zeros(64, np.int32), np.stack(mats))
    s.build_accel()
    org = np.zeros((30000, 4), np.float32)
    org[:, :3] = rng.uniform(-6, 6, (30000, 3))
    org[:, 3] = 1e-5
    dd = rng.normal(size=(30000, 3))
    d = np.zeros((30000, 4), np.float32)
    d[:, :3] = dd / np.linalg.norm(dd, axis=1, keepdims=True)
    d[:, 3] = np.inf
    g = gpu_closest(device, s, org, d)
    v, i, p = s.geometry()
    tl, tp, inst = s.tlas()
    o = O.trace_two_level(v, i, p, [s.blas(0)], inst, tl, tp, org, d)
    assert_same(g, o, keys=("t", "u", "v", "triangle", "instance", "node_tests", "triangle_tests"))


@pytest.mark.parametrize("kind", ["flat", "two_level"])
def test_origin_order_gives_identical_results(device, kind):
    """Large launches claim rays in origin-cell order; every output is the
    same as with input order (bit for bit, counters included)."""
    from yaoray_amd import native as N
    if kind == "flat":
        s = Scene.triangles(20000, seed=5)
    else:
        s = Scene.instanced(instances=200, subdivisions=2, variants=4, env_width=8, env_height=4, seed=6)
    s.build_accel()
    o1, d1 = random_rays(70000, seed=9)
    o1[:, :3] = o1[:, :3] * 3.0 - 1.0  # some origins outside the scene box
    o2, d2 = s.camera_rays(256, 128)
    org, d = np.concatenate([o1, o2]), np.concatenate([d1, d2])
    org[5, 0] = np.nan  # a NaN origin falls in the first cell and misses
    device.upload_scene(s)
    try:
        device.set_trace_order(N.TRACE_ORDER_INPUT)
        a = device.trace_closest(org, d, counters=True)
        aa = device.trace_any(org, d, counters=True)
        device.set_trace_order(N.TRACE_ORDER_ORIGIN)
        b = device.trace_closest(org, d, counters=True)
        bb = device.trace_any(org, d, counters=True)
    finally:
        device.set_trace_order(N.TRACE_ORDER_ORIGIN)
    assert_same(b, a, keys=("t", "u", "v", "triangle", "instance", "node_tests", "triangle_tests"))
    for k in ("occluded", "node_tests", "triangle_tests"):
        assert np.array_equal(bb[k], aa[k]), k
    assert b["triangle"][5] == -1
    assert 0.01 < (a["triangle"] >= 0).mean() < 1.0


def reciprocal_queries(device, z):
    """1 / z as the triangle test computes it, and whether the slab test agrees
    with that value as the entry distance: rays along (0, 0, z) from c = +-2^k
    away at the triangle (0,0,0) (1,0,0) (0,1,0), whose determinant is -z. The
    hit's t is c * fl(1/z), exact; the box, flat at z = 0, is entered at the same
    distance, so it is met with t_max there (one triangle test) and missed with
    the float below (none)."""
    z = np.ascontiguousarray(z, np.float32)
    with np.errstate(all="ignore"):
        r = np.float32(1.0) / z
        e = np.where(np.isfinite(r) & (r != 0.0), np.frexp(r)[1], 0)
        c = np.copysign(np.ldexp(np.float32(1.0), np.clip(-e, -126, 126)), z).astype(np.float32)
        at = (c * r).astype(np.float32)
    org, d = np.full((len(z), 4), 0.25, np.float32), np.zeros((len(z), 4), np.float32)
    org[:, 2], org[:, 3], d[:, 2] = -c, 0.0, z
    d[:, 3] = np.inf
    g = device.trace_closest(org, d, counters=True)
    met, missed = d.copy(), d.copy()
    met[:, 3], missed[:, 3] = at, np.nextafter(at, np.float32(0.0))
    m = device.trace_closest(org, met, counters=True)["triangle_tests"]
    n = device.trace_closest(org, missed, counters=True)["triangle_tests"]
    return at, g, m, n


def test_reciprocals_are_the_ieee_quotients(device):
    """The traversal's reciprocal equals float division bit for bit: all
    mantissas at both ends of its fast range, [2^-100, 2^100], just outside and
    inside, both signs; zeros, subnormals, infinities and NaN as the oracle.
    Determinants below 1e-8 are rejected whatever their reciprocal is, so
    smaller z show in the slab test only."""
    s = MeshArrays().add_triangles(np.array([[[0, 0, 0], [1, 0, 0], [0, 1, 0]]], np.float32)).scene()
    s.build_accel()
    device.upload_scene(s)
    mantissas = np.arange(1 << 23, dtype=np.uint32)
    for sign in (0, 1):
        for exponent in (-101, -100, -27, -1, 0, 99, 100, 127):
            z = (mantissas | np.uint32(exponent + 127 << 23) | np.uint32(sign << 31)).view(np.float32)
            at, g, met, missed = reciprocal_queries(device, z)
            assert (met == 1).all() and (missed == 0).all(), (sign, exponent)
            if exponent >= -26:
                assert (g["triangle"] == 0).all() and same_bits(g["t"], at), (sign, exponent)
    special = np.array([0.0, np.inf, np.nan, 1e-45, 2.0**-149 * 3, 2.0**-127, 2.0**-126, 2.0**-101, 2.0**101, 3.4e38], np.float32)
    z = np.tile(np.concatenate([special, -special]), 3)
    org, d = np.full((len(z), 4), 0.25, np.float32), np.zeros((len(z), 4), np.float32)
    org[:, 2], org[:, 3], d[:, 2], d[:, 3] = np.repeat([-1.0, 0.0, 1.0], 2 * len(special)), 0.0, z, np.inf
    v, i, p = s.geometry()
    assert_same(device.trace_closest(org, d, counters=True), O.trace_flat(v, i, p, s.flat_bvh(), org, d))
