"""Traversal of large queues, where a wave works through a run of rays and
refills its idle lanes, against the same render in passes small enough for one
ray a lane: the same image bit for bit, the same rays, node visits, triangle tests
and hits.  Sizes at the queue length from which runs are used, one path more or
less, and where the last wave's run is a remainder.
"""
import numpy as np
import pytest

from atrc_amd import capi, scenes

pytestmark = pytest.mark.gpu

RUNS_MIN = 1 << 21


def _render(W, H, spp, accel, stats, max_paths, monkeypatch):
    monkeypatch.setenv("AGX_MAX_PATHS", str(max_paths))
    s, _, tr = scenes.procedural_spheres(n_spheres=24, subdiv=3, seed=3, extent=20.0, sun=True)
    cam = {"pos": (-12.0, -16.0, 24.0), "dst": (10.0, 10.0, 8.0), "fov": 40.0}
    s.accel = accel
    desc, keep = s.to_desc()
    with capi.Context(0) as ctx:
        ctx.upload_scene(desc)
        p = scenes.render_params(W, H, spp, cam, seed=11, collect_stats=stats, **dict(tr, max_depth=4))
        return ctx.render(p)["image"], ctx.stats()


@pytest.mark.parametrize("accel", [capi.ACCEL_BVH4, capi.ACCEL_BVH4_WATERTIGHT])
@pytest.mark.parametrize("W,H,spp", [(2048, 1024, 1), (2047, 1025, 1), (683, 1025, 3), (1601, 1409, 2)])
def test_runs_change_nothing(W, H, spp, accel, monkeypatch):
    print(f"[runs] {W}x{H} {spp} spp, accel {accel}", flush=True)
    assert W * H * spp > RUNS_MIN - 4096
    a, sa = _render(W, H, spp, accel, True, 1 << 25, monkeypatch)
    b, sb = _render(W, H, spp, accel, True, 1 << 19, monkeypatch)
    np.testing.assert_array_equal(a.view(np.uint32), b.view(np.uint32))
    for k in ("closest_rays", "shadow_rays", "closest_node_visits", "closest_tri_tests", "closest_hits",
              "shadow_node_visits", "shadow_tri_tests"):
        assert sa[k] == sb[k], k
    c, _ = _render(W, H, spp, accel, False, 1 << 25, monkeypatch)
    np.testing.assert_array_equal(a.view(np.uint32), c.view(np.uint32))
