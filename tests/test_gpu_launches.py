"""The render loop's launch decisions: passes whose first bounce is thinned by
roulette (queues counted on the device), scenes without lights (no shadow
launches) and images of a few paths, path for path against the oracle; the ray
counts are those of the queues and the same in every pass split.
"""
import ctypes as C

import numpy as np
import pytest

from atrc_amd import capi, scenes
from oracle import py_oracle as po

from test_gpu_render_parity import _path_parity

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("accel", [capi.ACCEL_ATRC, capi.ACCEL_BVH4, capi.ACCEL_BVH4_WATERTIGHT])
@pytest.mark.parametrize("W,H", [(1, 1), (13, 5), (65, 63), (64, 64), (241, 17)])  # 4096: the one-block queues
@pytest.mark.parametrize("min_depth", [0, 2])
def test_small_images_path_parity(gpu_ctx, W, H, min_depth, accel):
    s, cam, tr = scenes.cornell_box()
    s.accel = accel
    # a single path may round to another decision: small images must agree on all but one
    _path_parity(gpu_ctx, s, cam, dict(tr, min_depth=min_depth), W, H, f"small {W}x{H} min_depth {min_depth}",
                 min_frac=min(0.97, 1 - 1.5 / (W * H)))


@pytest.mark.parametrize("accel", [capi.ACCEL_ATRC, capi.ACCEL_BVH4, capi.ACCEL_BVH4_WATERTIGHT])
@pytest.mark.parametrize("min_depth", [0, 2])
def test_images_of_one_path(gpu_ctx, min_depth, accel):
    """Renders of a single path: of forty samples, asked for one by one, all but one agree with the oracle."""
    s, cam, tr = scenes.cornell_box()
    s.accel = accel
    desc, keep = s.to_desc()
    gpu_ctx.upload_scene(desc)
    ref = po.OracleScene(desc, 32)
    print(f"[launches] one path, min_depth {min_depth}, accel {accel}", flush=True)
    off = lit = 0
    for k in range(40):
        p = scenes.render_params(1, 1, 1, cam, seed=1234, sample_begin=k, **dict(tr, min_depth=min_depth))
        g, r = gpu_ctx.render(p)["image"].astype(np.float64), ref.render(p, threads=1)["image"]
        off += bool((np.abs(g - r).max() > 1e-3 * (np.abs(r).max() + 1e-2)))
        lit += bool(r.any())
    assert off <= 1 and lit >= 10


def test_no_lights(gpu_ctx):
    s, cam, tr = scenes.cornell_box()
    s.entities[-1].emit = (0.0, 0.0, 0.0)
    s.accel = capi.ACCEL_BVH4
    desc, keep = s.to_desc()
    gpu_ctx.upload_scene(desc)
    print("[launches] cornell without its light", flush=True)
    g = gpu_ctx.render(scenes.render_params(40, 30, 4, cam, seed=3, **tr))
    st = gpu_ctx.stats()
    assert not g["image"].any() and st["shadow_rays"] == 0 and st["trace_shadow_launches"] == 0
    assert st["closest_rays"] > 40 * 30 * 4


def test_ray_counts_add_up(gpu_ctx):
    """The rays of one render are those of its samples rendered one at a time."""
    s, cam, tr = scenes.cornell_box()
    s.accel = capi.ACCEL_BVH4
    desc, keep = s.to_desc()
    gpu_ctx.upload_scene(desc)
    print("[launches] ray counts of 3 samples, together and apart", flush=True)
    acc = np.zeros(3, np.int64)
    for k in range(3):
        gpu_ctx.render(scenes.render_params(70, 51, 1, cam, seed=3, sample_begin=k, **tr))
        st = gpu_ctx.stats()
        acc += [st["closest_rays"], st["shadow_rays"], st["paths"]]
    gpu_ctx.render(scenes.render_params(70, 51, 3, cam, seed=3, **tr))
    st = gpu_ctx.stats()
    assert [st["closest_rays"], st["shadow_rays"], st["paths"]] == acc.tolist()


@pytest.mark.parametrize("media", [False, True])
def test_cancelled_renders_keep_their_times(gpu_ctx, media):
    """A render cancelled after its first bounce: the times of the kernels that ran
    are in its statistics, and the next render is a whole one."""
    s, cam, tr = scenes.volumetric_room(n_clutter_tris=2000, grid_n=16) if media else scenes.cornell_box()
    s.accel = capi.ACCEL_BVH4
    desc, keep = s.to_desc()
    gpu_ctx.upload_scene(desc)
    print(f"[launches] cancelled render, media {media}", flush=True)
    p = scenes.render_params(256, 256, 4, cam, seed=3, **tr)
    whole = gpu_ctx.render(p, aovs=False)["image"]
    full = gpu_ctx.stats()
    g = gpu_ctx.render(p, cancel=C.c_int32(1), aovs=False)
    st = gpu_ctx.stats()
    assert g["cancelled"] and not g["image"].any()
    assert st["trace_closest_launches"] == 1
    assert 0 < st["trace_closest_ms"] < full["trace_closest_ms"] and 0 < st["shade_ms"] < full["shade_ms"]
    assert st["trace_closest_ms"] + st["trace_shadow_ms"] + st["shade_ms"] <= 1.05 * st["total_ms"]
    np.testing.assert_array_equal(gpu_ctx.render(p, aovs=False)["image"], whole)
