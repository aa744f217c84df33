"""Ray-query parity: the gfx950 traversal against the CPU restatement of Atrc's
scene queries (oracle, FP32), ray for ray.

Bar: bit-exact.  Entity id, primitive id (original triangle index / quad half),
hit distance t and barycentrics (u, v) must be identical, and any-hit results
identical, because the GPU traverses the same Atrc BVHs with the same FP32
operation order (Möller–Trumbore, inclusive t bounds, last-tested wins ties:
src/tracer/include/agz/tracer/utility/triangle_aux.h:38-69,
src/tracer/src/core/geometry/triangle_bvh.cpp:403-488).

Every case runs in both acceleration modes.  AGX_ACCEL_ATRC also reproduces
Atrc's node visits and triangle tests.  AGX_ACCEL_BVH4 (SAH BVH4, near-first)
tests primitives in another order, so where two primitives are hit at exactly
the same t the other one may win: a ray whose result differs from the oracle
must then carry the oracle's t bit for bit (a tie), and such rays must be rare.
"""
import numpy as np
import pytest

from atrc_amd import capi, scenes
from oracle import py_oracle as po

from conftest import log

pytestmark = pytest.mark.gpu


@pytest.fixture(params=["atrc", "bvh4"])
def accel(request):
    return {"atrc": capi.ACCEL_ATRC, "bvh4": capi.ACCEL_BVH4}[request.param]


def _compare(gpu_ctx, scene, o, d, tmin, tmax, label, accel=capi.ACCEL_ATRC):
    scene.accel = accel
    desc, keep = scene.to_desc()
    gpu_ctx.upload_scene(desc)
    ref = po.OracleScene(desc, 32)
    mode = "atrc" if accel == capi.ACCEL_ATRC else "bvh4"
    log(f"[trace parity] {label} ({mode}): {len(o)} rays")
    g = gpu_ctx.trace_rays(o, d, tmin, tmax)
    r = ref.trace_rays(o, d, tmin, tmax)
    hit = r["entity"] >= 0
    st = gpu_ctx.stats()
    same = (g["entity"] == r["entity"]) & (g["prim"] == r["prim"])
    if accel == capi.ACCEL_ATRC:
        assert same.all()
    else:
        # a different winner only at exactly equal t: coplanar surfaces (the Cornell
        # boxes stand on the floor, so rays starting inside a box meet its bottom
        # face and the floor at the same t)
        diff = ~same
        log(f"  equal-t ties resolved differently: {int(diff.sum())}")
        assert diff.mean() < 1e-2
        np.testing.assert_array_equal(g["t"][diff].view(np.uint32), r["t"][diff].view(np.uint32))
        hit = hit & same
    # bit-exact FP32 distances and barycentrics
    np.testing.assert_array_equal(g["t"][hit].view(np.uint32), r["t"][hit].view(np.uint32))
    np.testing.assert_array_equal(g["u"][hit].view(np.uint32), r["u"][hit].view(np.uint32))
    np.testing.assert_array_equal(g["v"][hit].view(np.uint32), r["v"][hit].view(np.uint32))
    if accel == capi.ACCEL_ATRC:
        # same BVH, same order: node visits and triangle tests agree with the oracle
        assert st["closest_node_visits"] == r["counters"]["node_visits"]
        assert st["closest_tri_tests"] == r["counters"]["tri_tests"]
    else:
        log(f"  node visits / ray: bvh4 {st['closest_node_visits'] / len(o):.2f} (x4 boxes), "
            f"atrc {r['counters']['node_visits'] / len(o):.2f}; triangle tests / ray: bvh4 "
            f"{st['closest_tri_tests'] / len(o):.2f}, atrc {r['counters']['tri_tests'] / len(o):.2f}")
    ga = gpu_ctx.trace_rays(o, d, tmin, tmax, any_hit=True)
    ra = ref.trace_rays(o, d, tmin, tmax, any_hit=True)
    np.testing.assert_array_equal(ga["entity"], ra["entity"])
    return (r["entity"] >= 0).mean()


def test_cornell_rays(gpu_ctx, accel):
    s, _, _ = scenes.cornell_box()
    o, d = scenes.random_rays(((0.05, 0.05, 0.05), (5.5, 5.5, 5.5)), 200_000, seed=7)
    n = len(o)
    frac = _compare(gpu_ctx, s, o, d, np.zeros(n, np.float32), np.full(n, np.inf, np.float32), "cornell", accel)
    assert frac > 0.8  # the box is open at the front (y = 0)


def test_cornell_native_aggregate_and_bounded_rays(gpu_ctx, accel):
    s, _, _ = scenes.cornell_box()
    s.aggregate = capi.AGGREGATE_NATIVE
    o, d = scenes.random_rays(((0.05, 0.05, 0.05), (5.5, 5.5, 5.5)), 100_000, seed=8)
    rng = np.random.default_rng(9)
    tmin = rng.uniform(0, 0.5, len(o)).astype(np.float32)
    tmax = rng.uniform(0.5, 6.0, len(o)).astype(np.float32)
    _compare(gpu_ctx, s, o, d, tmin, tmax, "cornell/native/bounded", accel)


def test_procedural_mesh_rays(gpu_ctx, accel):
    s, _, _ = scenes.procedural_spheres(n_spheres=24, subdiv=3, seed=3, extent=20.0)
    o, d = scenes.random_rays(((-2, -2, -2), (22, 22, 22)), 200_000, seed=11)
    n = len(o)
    frac = _compare(gpu_ctx, s, o, d, np.zeros(n, np.float32), np.full(n, np.inf, np.float32), "spheres24", accel)
    assert frac > 0.3


def test_analytic_shapes_rays(gpu_ctx, accel):
    """Transformed triangle, sphere and disk entities (local-space intersection)."""
    s = scenes.Scene(aggregate=capi.AGGREGATE_BVH)
    m = s.add_material(scenes.Material(color=(0.5, 0.5, 0.5)))
    rot = np.array([[0.6, -0.8, 0.0], [0.8, 0.6, 0.0], [0.0, 0.0, 1.0]])
    for k in range(6):
        M = np.hstack([rot * (0.5 + 0.25 * k), np.array([[k * 2.0], [1.0], [0.5 * k]])])
        s.add(scenes.Entity(capi.GEOM_SPHERE, m, radius=1.0, local_to_world=tuple(M.reshape(-1))))
        s.add(scenes.Entity(capi.GEOM_DISK, m, radius=0.8, local_to_world=tuple((M + np.array(
            [[0, 0, 0, 0], [0, 0, 0, 3.0], [0, 0, 0, 0]])).reshape(-1))))
        s.add(scenes.Entity(capi.GEOM_TRIANGLE, m, points=((0, 0, 0), (1, 0, 0), (0, 1, 0)),
                            local_to_world=tuple((M + np.array([[0, 0, 0, 0], [0, 0, 0, -3.0], [0, 0, 0, 0]])).reshape(-1))))
    o, d = scenes.random_rays(((-2, -4, -2), (13, 6, 5)), 100_000, seed=12)
    n = len(o)
    _compare(gpu_ctx, s, o, d, np.zeros(n, np.float32), np.full(n, np.inf, np.float32), "analytic", accel)


def test_ray_replay_captures_every_query(gpu_ctx):
    """agx_debug_replay_rays captures exactly the queries the render issued."""
    s, cam, tr = scenes.cornell_box()
    s.accel = capi.ACCEL_BVH4
    desc, keep = s.to_desc()
    gpu_ctx.upload_scene(desc)
    p = scenes.render_params(64, 64, 2, cam, seed=5, **tr)
    rr = gpu_ctx.replay_rays(p)
    st = gpu_ctx.stats()
    log(f"[replay] cornell 64x64 2 spp: {rr}")
    assert rr["closest_rays"] == st["closest_rays"] and rr["shadow_rays"] == st["shadow_rays"]
    assert rr["replay_closest_ms"] > 0 and rr["replay_shadow_ms"] > 0


def test_ray_replay_times_are_the_renders_own(gpu_ctx):
    """The closest-hit and any-hit times that a replay reports of its render do
    not hold the capturing."""
    s, cam, tr = scenes.procedural_spheres(n_spheres=24, subdiv=3, seed=3, extent=20.0, sun=True)
    cam = {"pos": (-12.0, -16.0, 24.0), "dst": (10.0, 10.0, 8.0), "fov": 40.0}
    s.accel = capi.ACCEL_BVH4
    desc, keep = s.to_desc()
    gpu_ctx.upload_scene(desc)
    p = scenes.render_params(1024, 768, 2, cam, seed=5, **tr)
    plain, replay = [], []
    for _ in range(4):  # the first of each warms up; the fastest counts
        gpu_ctx.render(p, aovs=False)
        st = gpu_ctx.stats()
        plain.append((st["trace_closest_ms"], st["trace_shadow_ms"]))
        rr = gpu_ctx.replay_rays(p, max_rays=1 << 24, reps=1)
        replay.append((rr["render_closest_ms"], rr["render_shadow_ms"]))
    a, b = np.min(plain, axis=0), np.min(replay, axis=0)
    log(f"[replay] closest / any hit {a} ms in a render, {b} ms in a replay's")
    assert (b < 1.4 * a + 0.05).all()
