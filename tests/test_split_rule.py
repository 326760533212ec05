"""The automatic list split's count of stretches (host logic, CPU only)."""
import ctypes
import os
import subprocess

import pytest

SHIM = r"""
#include "4dzb_amd/csrc/fd_host.h"
extern "C" int segs(int w, int h, int ntris, int grid_log2, int waves, int req, int variant) {
    FdArgs a;
    const fdh::Model md{nullptr, 4, 3, nullptr, ntris};
    fdh::fill_args(a, md, nullptr, nullptr, w, h, FdLight{}, 0.0f, 0, grid_log2, 3, nullptr, nullptr, 1);
    a.occWaves = waves;
    a.occVariant = variant;
    fdh::apply_split(a, req);
    return a.segs;
}
"""


@pytest.fixture(scope="module")
def segs(fd, tmp_path_factory):
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    d = tmp_path_factory.mktemp("split")
    src, so = d / "shim.cpp", d / "shim.so"
    src.write_text(SHIM)
    fd.lib()
    subprocess.run(["g++", "-std=c++17", "-O1", "-w", "-fPIC", "-shared", "-D__HIP_PLATFORM_AMD__", f"-I{root}",
                    "-I/opt/rocm/include", str(src), "-o", str(so), fd.LIB_PATH,
                    f"-Wl,-rpath,{os.path.dirname(fd.LIB_PATH)}", "-Wl,--unresolved-symbols=ignore-in-shared-libs"],
                   check=True)
    f = ctypes.CDLL(str(so)).segs
    f.argtypes, f.restype = [ctypes.c_int] * 7, ctypes.c_int
    return lambda *a, variant=0: f(*a, variant)


@pytest.mark.parametrize("bins", [8, 16, 32])
@pytest.mark.parametrize("w", [1, 16, 64, 96, 128, 176, 512])
def test_small_views_of_dense_scenes_split(segs, bins, w):
    """A small view leaves the GPU idle however long its lists are: from 512
    triangles per bin on it gets as many stretches as its waves call for
    (whole lists there took 7271 us against 1674 for 20 spheres of 1M
    triangles at 176 x 176 receivers)."""
    nb = bins * bins
    slots = (w * w + 63) // 64 + nb + 1
    for waves in (4, 8):
        n = slots * waves
        most = max(1, min(16, 49152 // n)) if slots <= 2048 and n < 6144 else 1
        for per_bin in (512, 1000, 4000):
            assert segs(w, w, per_bin * nb, bins.bit_length() - 1, waves, 0) == most, (waves, per_bin)


def test_few_triangles_and_explicit_counts(segs):
    """At most 4 stretches below 16 triangles per bin, 8 below 512; explicit
    counts as asked; no triangles, one."""
    for per_bin, most in ((0, 4), (15, 4), (16, 8), (511, 8), (512, 16)):
        assert segs(64, 64, max(1, per_bin * 256), 4, 8, 0) == most, per_bin
    assert [segs(64, 64, 10 ** 6, 4, 8, s) for s in (1, 3, 64)] == [1, 3, 64]
    assert segs(64, 64, 0, 4, 8, 0) == 1 and segs(64, 64, 0, 4, 8, 7) == 1


def test_bin_queue_variant(segs):
    """The bin-queue variant's waves do not share a list: as many stretches as
    its waves call for, however few the triangles (1274 us with 8, 764 with 16:
    40 k evenly spread triangles over 96 x 96 receivers)."""
    for per_bin in (1, 15, 16, 156, 511, 512, 4000):
        for w in (48, 96, 160):
            slots = (w * w + 63) // 64 + 257
            assert segs(w, w, per_bin * 256, 4, 8, 0, variant=1) == min(16, 49152 // (8 * slots)), (per_bin, w)
    assert segs(96, 96, 40000, 4, 8, 3, variant=1) == 3
