"""The quad rasteriser's single-precision bounds on the CPU: random cameras
(frames of 1 to 16384 pixels, 0.2 to 178 degrees, eyes in the scene and up to
2^20 voxels off) and quads that a pixel's ray just hits.  The bounds decide only
what is left out, so a hit outside one would be a pixel drawn wrong.  The
functions are cut from mesoengine_amd/csrc/raster.hip; the reciprocal
instruction is one unit off either way at random."""
import os
import subprocess

import pytest

from test_native_walks import CLANG, CLANGXX, CSRC, INSTRUCTIONS, ROOT

pytestmark = pytest.mark.skipif(not (os.path.exists(CLANGXX) and os.path.exists(CLANG)),
                                reason="ROCm clang not installed")


def _cut(text, first, last):
    """from the line that starts with `first` up to the one that starts with `last`"""
    a = text.index("\n" + first) + 1
    return text[a:text.index("\n" + last, a) + 1]


@pytest.fixture(scope="module")
def bounds(tmp_path_factory):
    tmp = tmp_path_factory.mktemp("bounds")
    text = open(os.path.join(CSRC, "traverse.h")).read()
    for ins, host in INSTRUCTIONS.items():
        text = text.replace(ins, host)
    text = text.replace('#include "meso_internal.h"',
                        '#include "%s"' % os.path.join(CSRC, "meso_internal.h"))
    (tmp / "traverse_host.h").write_text(text)
    raster = open(os.path.join(CSRC, "raster.hip")).read()
    host = (_cut(raster, "struct QuadGeom {", "__device__ __forceinline__ QuadGeom quad_decode") +
            _cut(raster, "__device__ __forceinline__ float pick3", "// t of the hit on the quad") +
            _cut(raster, "__device__ __forceinline__ float quad_hit", "// conservative pixel rect") +
            "constexpr int kSmall = 64;\n" +
            _cut(raster, "struct RasterView {", "// One shell's pixel tests") +
            _cut(raster, "__device__ __forceinline__ float square_dist",
                 "__global__ void __launch_bounds__(256) raster_begin_kernel"))
    (tmp / "raster_bounds_host.h").write_text(host)
    exe = str(tmp / "raster_bounds")
    subprocess.check_call([CLANGXX, "-std=c++17", "-D__HIP_PLATFORM_AMD__", "-w", "-O2",
                           "-ffp-contract=off", "-I", str(tmp), "-I/opt/rocm/include",
                           os.path.join(ROOT, "tests", "native", "raster_bounds.cpp"), "-o", exe])
    return exe


@pytest.mark.parametrize("seed", [1, 2, 3])
def test_every_hit_is_in_bounds(bounds, seed):
    r = subprocess.run([bounds, str(seed), "40000"], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stdout[-2000:] + r.stderr[-2000:]
