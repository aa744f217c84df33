"""Quads in the BVH4 mode, whose records carry their first triangle, against
the oracle ray for ray: planar and twisted quads, quads of which one half is
degenerate (B = A leaves no first triangle and goes through the entity), and
coplanar overlapping quads whose ties the aggregate's order decides; rays at
random and aimed at corners, edges and the shared diagonal.  (The native
aggregate: Atrc's entity BVH culls by unpadded boxes and loses some of the rays
aimed exactly at the edges of flat boxes.)
"""
import numpy as np
import pytest

from atrc_amd import capi, scenes
from oracle import py_oracle as po

pytestmark = pytest.mark.gpu

QUADS = {
    "planar": [((0, 0, 0), (1, 0, 0), (1, 1, 0), (0, 1, 0)), ((0.3, 0.2, 0.5), (1.4, 0.1, 0.7), (1.5, 1.3, 0.9),
                                                             (0.4, 1.4, 0.7))],
    "twisted": [((0, 0, 0), (1, 0, 0.4), (1, 1, 0), (0, 1, 0.4)), ((0, 0, 1), (1, 0.2, 0.8), (0.9, 1, 1.3), (0, 1, 1))],
    "no_first_half": [((0, 0, 0), (0, 0, 0), (1, 1, 0), (0, 1, 0)), ((0, 0, 1), (1, 0, 1), (1, 1, 1), (0, 1, 1))],
    "no_second_half": [((0, 0, 0), (1, 0, 0), (1, 1, 0), (1, 1, 0)), ((0, 0, 1), (1, 0, 1), (1, 1, 1), (0, 1, 1))],
    "coplanar": [((0, 0, 0), (1, 0, 0), (1, 1, 0), (0, 1, 0)), ((0.25, 0.25, 0), (1.25, 0.25, 0), (1.25, 1.25, 0),
                                                                (0.25, 1.25, 0)),
                 ((0, 0, 0), (0, 1, 0), (1, 1, 0), (1, 0, 0))],
}


@pytest.mark.parametrize("which", sorted(QUADS))
def test_quads_match_the_oracle(gpu_ctx, which):
    s = scenes.Scene(aggregate=capi.AGGREGATE_NATIVE, accel=capi.ACCEL_BVH4)
    m = s.add_material(scenes.Material(color=(0.5, 0.5, 0.5)))
    for q in QUADS[which]:
        s.add(scenes.Entity(capi.GEOM_QUAD, m, points=q))
    s.add(scenes.Entity(capi.GEOM_SPHERE, m, radius=0.2, local_to_world=(1, 0, 0, 0.5, 0, 1, 0, 0.5, 0, 0, 1, 0.3)))
    rng = np.random.default_rng(3)
    o, d = scenes.random_rays(((-1, -1, -1), (2, 2, 2)), 6000, seed=4)
    pts = []
    for q in QUADS[which]:
        a, b, c, e = np.asarray(q, np.float32)
        k = rng.choice([0.0, 0.25, 0.5, 1.0], (200, 1)).astype(np.float32)
        pts += [a + (c - a) * k, a + (b - a) * k, c + (e - c) * k]  # the diagonal and two edges
    pts = np.concatenate(pts)
    oo = rng.uniform(-1, 2, pts.shape).astype(np.float32)
    oo[:, 2] += np.float32(3) * rng.choice([-1, 1], len(oo)).astype(np.float32)
    o, d = np.concatenate([o, oo]), np.concatenate([d, (pts - oo).astype(np.float32)])
    n = len(o)
    tmin, tmax = np.zeros(n, np.float32), np.full(n, np.inf, np.float32)
    desc, keep = s.to_desc()
    gpu_ctx.upload_scene(desc)
    ref = po.OracleScene(desc, 32)
    print(f"[quads] {which}", flush=True)
    g, r = gpu_ctx.trace_rays(o, d, tmin, tmax), ref.trace_rays(o, d, tmin, tmax)
    for k in ("entity", "prim"):
        np.testing.assert_array_equal(g[k], r[k])
    hit = r["entity"] >= 0
    for k in ("t", "u", "v"):
        np.testing.assert_array_equal(g[k][hit].view(np.uint32), r[k][hit].view(np.uint32))
    ga, ra = gpu_ctx.trace_rays(o, d, tmin, tmax, any_hit=True), ref.trace_rays(o, d, tmin, tmax, any_hit=True)
    np.testing.assert_array_equal(ga["entity"], ra["entity"])
