"""Traversal of large queues, where a wave works through a run of rays and
refills its idle lanes, against the same render in passes small enough for one
ray a lane: the same image bit for bit, the same rays, node visits, triangle tests
and hits.  Passes at the queue length from which runs are used, one path less and
one more, and where the last wave's run is a remainder; trees for the small and
for the large traversal stack.  The statistics tell which kernels ran.
"""
import numpy as np
import pytest

from atrc_amd import capi, scenes

pytestmark = pytest.mark.gpu

RUNS_MIN = 1 << 21


def _deep():
    """Triangles that shrink by a constant factor towards the origin: a tree of more than 21 levels, which takes the
    large stack."""
    k = 12.0 * 0.7 ** np.arange(300)[:, None]
    tri = np.stack([k * [1, 0, 0], k * [1.2, 0.1, 0], k * [1, 0.1, 0.2]], axis=1).reshape(-1, 3)
    return scenes.mesh_from_indexed(tri, np.tile([0.0, 0.0, 1.0], (len(tri), 1)), np.arange(len(tri)).reshape(-1, 3))


def _render(W, H, spp, accel, stats, max_paths, monkeypatch, deep=False, max_depth=4):
    monkeypatch.setenv("AGX_MAX_PATHS", str(max_paths))
    s, _, tr = scenes.procedural_spheres(n_spheres=24, subdiv=3, seed=3, extent=20.0, sun=True)
    cam = {"pos": (-12.0, -16.0, 24.0), "dst": (10.0, 10.0, 8.0), "fov": 40.0}
    s.accel = accel
    if deep:
        s.add(scenes.Entity(capi.GEOM_TRIANGLE_BVH, 0, tris=_deep()))
    desc, keep = s.to_desc()
    assert (capi.debug_scene_summary(desc)["bvh4_depth"] > 21) == deep
    with capi.Context(0) as ctx:
        ctx.upload_scene(desc)
        p = scenes.render_params(W, H, spp, cam, seed=11, collect_stats=stats, **dict(tr, max_depth=max_depth))
        return ctx.render(p)["image"], ctx.stats()


# 6223 x 337 = 2^21 - 1 paths, 5419 x 387 = 2^21 + 1
@pytest.mark.parametrize("accel", [capi.ACCEL_BVH4, capi.ACCEL_BVH4_WATERTIGHT])
@pytest.mark.parametrize("W,H,spp,deep", [(2048, 1024, 1, False), (6223, 337, 1, False), (5419, 387, 1, False),
                                          (2047, 1025, 1, False), (683, 1025, 3, False), (1601, 1409, 2, False),
                                          (5419, 387, 1, True)])
def test_runs_change_nothing(W, H, spp, deep, accel, monkeypatch):
    print(f"[runs] {W}x{H} {spp} spp, accel {accel}, deep {deep}", flush=True)
    a, sa = _render(W, H, spp, accel, True, 1 << 25, monkeypatch, deep)
    b, sb = _render(W, H, spp, accel, True, 1 << 19, monkeypatch, deep)
    np.testing.assert_array_equal(a.view(np.uint32), b.view(np.uint32))
    for k in ("closest_rays", "shadow_rays", "closest_node_visits", "closest_tri_tests", "closest_hits",
              "shadow_node_visits", "shadow_tri_tests"):
        assert sa[k] == sb[k], k
    c, sc = _render(W, H, spp, accel, False, 1 << 25, monkeypatch, deep)
    np.testing.assert_array_equal(a.view(np.uint32), c.view(np.uint32))
    # the first bounce's closest hits, and both traversals of at least the second
    assert sa["run_launches"] == sc["run_launches"] >= 2 + (W * H * spp >= RUNS_MIN)
    assert sb["run_launches"] == 0


@pytest.mark.parametrize("accel", [capi.ACCEL_BVH4, capi.ACCEL_BVH4_WATERTIGHT])
def test_runs_begin_at_their_queue_length(accel, monkeypatch):
    """The camera rays of 2^21 + 1 paths are traced in runs, those of 2^21 - 1 are not."""
    print(f"[runs] the limit, accel {accel}", flush=True)
    at, below = (_render(W, H, 1, accel, False, 1 << 25, monkeypatch, max_depth=1)[1]["run_launches"]
                 for W, H in ((5419, 387), (6223, 337)))
    assert at == below + 1


def test_runs_are_for_the_bvh4_modes(monkeypatch):
    s, cam, tr = scenes.cornell_box()
    s.accel = capi.ACCEL_ATRC
    desc, keep = s.to_desc()
    print("[runs] Atrc's structures", flush=True)
    with capi.Context(0) as ctx:
        ctx.upload_scene(desc)
        ctx.render(scenes.render_params(2048, 1024, 1, cam, seed=1, **dict(tr, max_depth=1)), aovs=False)
        assert ctx.stats()["run_launches"] == 0
