"""The image of a render is the same bit for bit whichever planes the caller
takes: without albedo, normal and denoise the path state and the film hold the
image alone."""
import numpy as np
import pytest

from atrc_amd import capi, scenes

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kw", [{}, {"filter": "gaussian", "filter_radius": 1.5, "filter_alpha": 2.0},
                                {"min_depth": 0}, {"use_mis": False}])
@pytest.mark.parametrize("scene", ["cornell", "delta", "fog"])
def test_image_does_not_depend_on_planes(gpu_ctx, scene, kw):
    s, cam, tr = {"cornell": scenes.cornell_box, "delta": lambda: scenes.cornell_delta(True),
                  "fog": lambda: scenes.volumetric_cornell(grid_n=8)}[scene]()
    s.accel = capi.ACCEL_BVH4
    desc, keep = s.to_desc()
    gpu_ctx.upload_scene(desc)
    print(f"[planes] {scene} {kw}", flush=True)
    p = scenes.render_params(61, 43, 3, cam, seed=21, **{**tr, **kw})
    image, full = gpu_ctx.render(p, aovs=False)["image"], gpu_ctx.render(p)
    np.testing.assert_array_equal(image.view(np.uint32), full["image"].view(np.uint32))
    again = gpu_ctx.render(p)
    for k in ("image", "albedo", "normal", "denoise"):
        np.testing.assert_array_equal(again[k].view(np.uint32), full[k].view(np.uint32))
    assert full["denoise"].max() > 0 and np.abs(full["normal"]).max() > 0.5
