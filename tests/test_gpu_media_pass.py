"""Tracking through media in a pass of its own, path for path against the
oracle where its branches meet their edges: grids one, two and odd numbers of
texels wide (the paired texel fetch), FP16 and FP32 texels, every wrap mode, a
scattering count that runs out, two lights of which one is hidden from most
points (occluded segments advance the stream without lookups), and bounded
media of two kinds met by lanes of one wave.
"""
import numpy as np
import pytest

from atrc_amd import capi, scenes

from test_gpu_render_parity import _path_parity

pytestmark = pytest.mark.gpu


def _scene(shape, f16, wrap, linear, max_scat):
    s, cam, tr = scenes.volumetric_cornell(grid_n=4)
    rng = np.random.default_rng(sum(shape) + wrap)
    g = rng.uniform(0.0, 2.0, shape)
    g = g.astype(np.float16).astype(np.float32) if f16 else (g / 3.0).astype(np.float32)
    het = s.media[1]
    # the texture is repeated or mirrored over twice the box, off its own centre
    het.density = scenes.Texture3D(grid=g, linear=linear, wrap=(wrap,) * 3,
                                   transform=(2.0, 0, 0, -0.3, 0, 1.5, 0, 0.1, 0, 0, -1.0, 0.9))
    het.max_scattering_count = max_scat
    s.media[0].max_scattering_count = max_scat
    # a second light, low behind the tall box: hidden from most of the room
    black = s.add_material(scenes.Material(kind=capi.MAT_IDEAL_BLACK))
    s.add(scenes.Entity(capi.GEOM_QUAD, black, emit=(9.0, 3.0, 6.0),
                        points=((5.0, 5.0, 0.4), (5.0, 5.4, 0.4), (4.8, 5.4, 0.9), (4.8, 5.0, 0.9))))
    s.accel = capi.ACCEL_BVH4
    return s, cam, dict(tr, max_depth=6)


@pytest.mark.parametrize("shape,f16,wrap,linear,max_scat", [
    ((1, 1, 1), True, capi.WRAP_CLAMP, True, 100),
    ((3, 2, 1), False, capi.WRAP_REPEAT, True, 100),
    ((1, 3, 2), True, capi.WRAP_MIRROR, True, 2),
    ((4, 3, 2), False, capi.WRAP_CLAMP, True, 1),
    ((5, 6, 7), True, capi.WRAP_REPEAT, True, 100),
    ((5, 6, 7), False, capi.WRAP_MIRROR, True, 3),
    ((6, 5, 9), True, capi.WRAP_CLAMP, False, 2),
])
def test_media_pass_path_parity(gpu_ctx, shape, f16, wrap, linear, max_scat):
    s, cam, tr = _scene(shape, f16, wrap, linear, max_scat)
    _path_parity(gpu_ctx, s, cam, tr, 96, 96, f"media pass, grid {shape} f16={f16} wrap={wrap} linear={linear}")
