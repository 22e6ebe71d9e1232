"""The quad rasteriser's list counter (mesoengine_amd/csrc/raster_lists.h)
replayed on the CPU past the capacity of its fields (2^24 records, 2^40 tests),
in small and in very many lots: neither field wraps, and the lots that are
listed fill the lists from their start without gaps.  And how a quad's pixels
are cut into tests: each in one, and never so many that a lot is refused."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "mesoengine_amd", "csrc")


@pytest.fixture(scope="module")
def replay(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("raster") / "replay")
    subprocess.check_call(["g++", "-std=c++17", "-O2", "-D__HIP_PLATFORM_AMD__", "-w", "-I", CSRC,
                           "-I/opt/rocm/include",
                           os.path.join(ROOT, "tests", "native", "raster_lists_replay.cpp"),
                           "-o", exe])
    return exe


@pytest.mark.parametrize("quads,groups,records,windows,area", [
    (24_000_000, 512, 1 << 22, 1 << 23, 12),       # a large culled pool seen from outside
    (2 ** 32 - 1, 512, 1 << 22, 1 << 23, 100),     # all the quads that a pool may hold
    (2 ** 32 - 1, 2048, 1 << 22, 1 << 23, 4000),
    (40_000_000, 2048, 1 << 22, 1 << 23, 1 << 28),  # quads of whole frames
    (100_000, 3, 700, 1 << 23, 50),
    (100_000, 512, 1 << 22, 3, 50),
    (100_000, 512, 0, 0, 50),
    (1, 1, 1, 1, 1)])
@pytest.mark.parametrize("seed", [1, 2])
def test_fields_never_wrap(replay, seed, quads, groups, records, windows, area):
    r = subprocess.run([replay] + [str(v) for v in (seed, quads, groups, records, windows, area)],
                       capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stdout + r.stderr


@pytest.mark.parametrize("seed", [1, 2, 3])
def test_rectangles_are_cut_into_tests(replay, seed):
    r = subprocess.run([replay, "cut", str(seed), "4000"], capture_output=True, timeout=120)
    assert r.returncode == 0
