"""What a render's path buffers take of the device's memory is what the pass size
reckons with, in scenes with many lights and with media.
"""
import ctypes as C
import subprocess
from pathlib import Path

import pytest

from atrc_amd import capi, scenes

pytestmark = pytest.mark.gpu

CSRC = Path(__file__).resolve().parent.parent / "atrc_amd" / "csrc"


@pytest.fixture(scope="module")
def path_bytes(tmp_path_factory):
    d = tmp_path_factory.mktemp("budget")
    (d / "budget.cpp").write_text('#include "agx_budget.h"\n#include <cstdio>\n#include <cstdlib>\nint main(int, char **a) '
                                  '{ std::printf("%zu", agx::path_bytes(std::atoi(a[1]), std::atoi(a[2]) != 0)); }\n')
    subprocess.run(["g++", "-std=c++17", f"-I{CSRC}", "-o", str(d / "budget"), str(d / "budget.cpp")], check=True)
    return lambda lights, media: int(subprocess.run([str(d / "budget"), str(lights), str(int(media))], check=True,
                                                    capture_output=True, timeout=20).stdout)


def _free():
    hip = C.CDLL("libamdhip64.so")
    free, total = C.c_size_t(), C.c_size_t()
    assert hip.hipMemGetInfo(C.byref(free), C.byref(total)) == 0
    return free.value


@pytest.mark.parametrize("media", [False, True])
@pytest.mark.parametrize("lights", [2, 16])
def test_path_buffers(path_bytes, lights, media, monkeypatch):
    n = 1 << 21
    monkeypatch.setenv("AGX_MAX_PATHS", str(n))
    s, cam, tr = scenes.volumetric_cornell(grid_n=8) if media else scenes.cornell_box()
    s.accel = capi.ACCEL_BVH4
    m = s.add_material(scenes.Material(kind=capi.MAT_IDEAL_BLACK))
    desc, keep = s.to_desc()
    more = lights - capi.debug_scene_summary(desc)["lights"]
    for k in range(more):
        x = 0.3 + 0.3 * k
        s.add(scenes.Entity(capi.GEOM_QUAD, m, points=((x, 1, 5.4), (x + 0.1, 1, 5.4), (x + 0.1, 1.1, 5.4), (x, 1.1, 5.4)),
                            emit=(1.0, 1.0, 1.0)))
    desc, keep = s.to_desc()
    assert capi.debug_scene_summary(desc)["lights"] == lights
    want = path_bytes(lights, media)
    with capi.Context(0) as ctx:
        ctx.upload_scene(desc)
        ctx.render(scenes.render_params(8, 8, 1, cam, seed=1, **tr), aovs=False)  # what a first render makes besides
        before = _free()
        # 1024 x 1024 at 2 samples: one pass of n paths; 84 bytes of film and 40 of planes a pixel
        ctx.render(scenes.render_params(1024, 1024, 2, cam, seed=1, **tr), aovs=False)
        used = (before - _free() - (1 << 20) * 124) / n
    print(f"[path memory] {lights} lights, media {media}: {used:.1f} bytes a path, reckoned {want}", flush=True)
    assert 0.97 * want - 8 < used < want + 8  # the allocator's granularity: 2 MB a buffer, some 30 buffers
