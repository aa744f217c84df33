"""The BVH4 box test never culls a triangle that the ray meets: rays for which
the reciprocal direction or the offset to a node is extreme, against the
brute force over every triangle (oracle, Moller-Trumbore as Atrc tests it).

The box test evaluates plane distances as q (step / d) + (origin - o) / d, so
the cases are those where these terms are zero, huge or cancel: directions
with one or two components that are zero (either sign) or of 1e-30, origins a
thousand scene sizes away, origins on vertex coordinates, directions that are
not of unit length.  Rays are aimed at points inside triangles and compared
where the brute force's hit lies inside its triangle by 2 %: at such a hit the
triangle test's own rounding cannot put the hit outside the triangle's box.
"""
import numpy as np
import pytest

from atrc_amd import capi, scenes
from oracle import py_oracle as po

pytestmark = pytest.mark.gpu


def _soup():
    pos, faces = scenes.icosphere(3)
    out = []
    for k, (r, c) in enumerate([(1.0, (0.0, 0.0, 0.0)), (0.37, (1.9, 0.4, -0.6)), (0.6, (-0.8, 2.1, 1.1))]):
        out.append(scenes.mesh_from_indexed(pos * r + np.array(c), pos, faces))
    return out


def _rays(kind, tris, n):
    rng = np.random.default_rng(17)
    b = rng.dirichlet((2.0, 2.0, 2.0), n)
    p = np.einsum("nk,nkd->nd", b, tris[rng.integers(0, len(tris), n)].astype(np.float64))  # points inside triangles
    d = rng.normal(size=(n, 3))
    if kind == "axis":
        d = np.zeros((n, 3))
        d[np.arange(n), rng.integers(0, 3, n)] = rng.choice([-1.0, 1.0], n)
        d = d * np.float32(1) * rng.choice([-1.0, 1.0], (n, 1))
    elif kind == "plane":  # one component zero, of either sign
        d[np.arange(n), rng.integers(0, 3, n)] = rng.choice([-0.0, 0.0], n)
    elif kind == "tiny":
        d[np.arange(n), rng.integers(0, 3, n)] = rng.choice([-1e-30, 1e-30, 1e-42], n)
    d /= np.linalg.norm(d, axis=1, keepdims=True)
    dist = {"far": 3000.0}.get(kind, 3.0)
    o = p - d * dist * rng.uniform(0.2, 1.0, (n, 1))
    if kind == "vertex":  # origins that share coordinates with bounds
        o = tris[rng.integers(0, len(tris), n), 0].astype(np.float64) * rng.choice([1.0, 1.0, 0.0], (n, 3))
        d = p - o
    if kind == "scaled":
        d = d * 10.0 ** rng.uniform(-6, 6, (n, 1))
    return o.astype(np.float32), d.astype(np.float32)


@pytest.mark.parametrize("accel", [capi.ACCEL_BVH4, capi.ACCEL_BVH4_WATERTIGHT])
@pytest.mark.parametrize("kind", ["axis", "plane", "tiny", "far", "vertex", "scaled"])
def test_box_test_is_conservative(gpu_ctx, kind, accel):
    meshes = _soup()
    s = scenes.Scene(aggregate=capi.AGGREGATE_BVH, accel=accel)
    m = s.add_material(scenes.Material(color=(0.5, 0.5, 0.5)))
    for t in meshes:
        s.add(scenes.Entity(capi.GEOM_TRIANGLE_BVH, m, tris=t))
    desc, keep = s.to_desc()
    gpu_ctx.upload_scene(desc)
    tris = np.concatenate([t[:, :3].reshape(-1, 3, 3) for t in meshes])
    o, d = _rays(kind, tris, 4000)
    n = len(o)
    tmin, tmax = np.full(n, 1e-3, np.float32), np.full(n, np.inf, np.float32)
    print(f"[box test] {kind}, accel {accel}", flush=True)
    prim, t, u, v = po.triangle_soup_closest(tris, o, d, tmin, tmax, watertight=accel == capi.ACCEL_BVH4_WATERTIGHT)
    inside = (prim >= 0) & (u > 0.02) & (v > 0.02) & (u + v < 0.98)
    assert inside.mean() > 0.5
    g = gpu_ctx.trace_rays(o, d, tmin, tmax)
    np.testing.assert_array_equal(g["t"][inside].view(np.uint32), t[inside].view(np.uint32))
    a = gpu_ctx.trace_rays(o, d, tmin, tmax, any_hit=True)
    assert (a["entity"][inside] == 1).all()


@pytest.mark.parametrize("accel", [capi.ACCEL_BVH4, capi.ACCEL_BVH4_WATERTIGHT])
@pytest.mark.parametrize("kind", ["any", "plane", "axis"])
@pytest.mark.parametrize("scale", [1e-33, 1e-25, 1e-20, 1e-12, 1e-9, 1e20, 1e30])
def test_length_of_the_direction(gpu_ctx, kind, scale, accel):
    """Rays whose whole direction is short or long, with and without zero
    components: the same hits as by brute force (distances are in units of it)."""
    meshes = _soup()
    s = scenes.Scene(aggregate=capi.AGGREGATE_BVH, accel=accel)
    m = s.add_material(scenes.Material(color=(0.5, 0.5, 0.5)))
    for t in meshes:
        s.add(scenes.Entity(capi.GEOM_TRIANGLE_BVH, m, tris=t))
    desc, keep = s.to_desc()
    gpu_ctx.upload_scene(desc)
    tris = np.concatenate([t[:, :3].reshape(-1, 3, 3) for t in meshes])
    o, d = _rays(kind, tris, 3000)
    d = (d.astype(np.float64) * scale).astype(np.float32)
    n = len(o)
    tmin, tmax = np.full(n, 1e-3 / scale, np.float32), np.full(n, np.inf, np.float32)
    print(f"[box test] {kind}, length {scale}, accel {accel}", flush=True)
    prim, t, u, v = po.triangle_soup_closest(tris, o, d, tmin, tmax, watertight=accel == capi.ACCEL_BVH4_WATERTIGHT)
    inside = (prim >= 0) & (u > 0.02) & (v > 0.02) & (u + v < 0.98)
    assert inside.mean() > 0.5
    g = gpu_ctx.trace_rays(o, d, tmin, tmax)
    np.testing.assert_array_equal(g["t"][inside].view(np.uint32), t[inside].view(np.uint32))
    a = gpu_ctx.trace_rays(o, d, tmin, tmax, any_hit=True)
    assert (a["entity"][inside] == 1).all()


@pytest.mark.parametrize("accel", [capi.ACCEL_BVH4, capi.ACCEL_BVH4_WATERTIGHT])
def test_directions_without_length(gpu_ctx, accel):
    """Zero and NaN directions hit nothing."""
    s = scenes.Scene(aggregate=capi.AGGREGATE_BVH, accel=accel)
    m = s.add_material(scenes.Material(color=(0.5, 0.5, 0.5)))
    for t in _soup():
        s.add(scenes.Entity(capi.GEOM_TRIANGLE_BVH, m, tris=t))
    desc, keep = s.to_desc()
    gpu_ctx.upload_scene(desc)
    o = np.random.default_rng(3).uniform(-1, 2, (300, 3)).astype(np.float32)
    d = np.zeros_like(o)
    d[100:] = np.nan
    d[200:, 0] = 1.0
    tmin, tmax = np.zeros(300, np.float32), np.full(300, np.inf, np.float32)
    print(f"[box test] zero and NaN directions, accel {accel}", flush=True)
    assert (gpu_ctx.trace_rays(o, d, tmin, tmax)["entity"] == -1).all()
    assert (gpu_ctx.trace_rays(o, d, tmin, tmax, any_hit=True)["entity"] == -1).all()
