"""The raymarcher's device walks (mesoengine_amd/csrc/traverse.h) run on the
CPU against the oracle, under ASan + UBSan (tests/native/traverse_walks.cpp).

The header is compiled for the host as it stands, but for its inline
instructions, which are replaced here by the same operations in C++.  What is
looked for above all is a read outside the scene, which must not be tried out
on a GPU: origins of secondary rays that rounding has put outside the scene,
as eyes far away give.
"""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "mesoengine_amd", "csrc")
ORACLE = os.path.join(ROOT, "oracle")
CLANG = "/opt/rocm/llvm/bin/clang"
CLANGXX = "/opt/rocm/llvm/bin/clang++"

pytestmark = pytest.mark.skipif(not (os.path.exists(CLANGXX) and os.path.exists(CLANG)),
                                reason="ROCm clang not installed")

# instruction -> what it computes (the float-to-integer conversions saturate)
INSTRUCTIONS = {
    'asm("v_med3_i32 %0, %1, %2, %3" : "=v"(m) : "v"(a), "v"(b), "v"(c));':
        "m = std::max(std::min(a, b), std::min(std::max(a, b), c));",
    'asm("v_cvt_flr_i32_f32 %0, %1" : "=v"(r) : "v"(x));':
        "r = x != x ? 0 : x >= 2147483648.0f ? 2147483647 : x < -2147483648.0f ? -2147483647 - 1"
        " : (int32_t)std::floor(x);",
    'asm("v_bfm_b32 %0, %1, 0" : "=v"(m) : "v"(k));': "m = (int32_t)((1u << k) - 1u);",
    'asm("v_xad_u32 %0, %1, -1, %2" : "=v"(r) : "v"(a), "v"(b));':
        "r = (int32_t)(~(uint32_t)a + (uint32_t)b);",
    'asm("" : "+v"(um[a]));': "",
}


@pytest.fixture(scope="module")
def walks(tmp_path_factory):
    tmp = tmp_path_factory.mktemp("walks")
    text = open(os.path.join(CSRC, "traverse.h")).read()
    for ins, host in INSTRUCTIONS.items():
        assert text.count(ins) == 1, ins
        text = text.replace(ins, host)
    assert "asm(" not in text
    text = text.replace('#include "meso_internal.h"',
                        '#include "%s"' % os.path.join(CSRC, "meso_internal.h"))
    (tmp / "traverse_host.h").write_text(text)
    san = ["-O1", "-g", "-ffp-contract=off", "-fsanitize=address,undefined",
           "-fno-sanitize=float-cast-overflow,shift,signed-integer-overflow",
           "-fno-sanitize-recover=undefined"]
    obj = str(tmp / "oracle.o")
    subprocess.check_call([CLANG, "-std=c11"] + san +
                          ["-c", os.path.join(ORACLE, "meso_oracle.c"), "-o", obj])
    exe = str(tmp / "traverse_walks")
    subprocess.check_call([CLANGXX, "-std=c++17", "-D__HIP_PLATFORM_AMD__", "-w"] + san +
                          ["-I", str(tmp), "-I", ORACLE, "-I/opt/rocm/include",
                           os.path.join(ROOT, "tests", "native", "traverse_walks.cpp"), obj,
                           "-o", exe, "-lm", "-lpthread"])
    return exe


def _run(walks, *args):
    r = subprocess.run([walks] + [str(a) for a in args], capture_output=True, text=True,
                       timeout=600)
    assert r.returncode == 0, r.stdout[-2000:] + r.stderr[-4000:]


@pytest.mark.parametrize("seed", [1, 2])
def test_parts_of_dense_rays(walks, seed):
    _run(walks, "dense", seed, 1_500_000)


@pytest.mark.parametrize("seed", [1, 2])
def test_secondary_rays_of_brick_scenes(walks, seed):
    _run(walks, "bricks", seed, 3_000_000)
