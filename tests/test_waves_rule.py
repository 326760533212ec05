"""Default waves per occlusion work item (host logic, CPU only)."""
import ctypes
import importlib
import os
import subprocess

import pytest

SHIM = r"""
#include "4dzb_amd/csrc/fd_host.h"
extern "C" int waves(int w, int h, int res, int grid_log2) {
    FdArgs a;
    const fdh::Model md{nullptr, 4, 3, nullptr, 1};
    fdh::fill_args(a, md, nullptr, nullptr, w, h, FdLight{}, 0.0f, 0, grid_log2, 3, nullptr, nullptr, 1);
    return fd_default_waves(res > 32 ? 2 : 1, a.chunkSlots);
}
"""


@pytest.fixture(scope="module")
def shim(fd, tmp_path_factory):
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    d = tmp_path_factory.mktemp("waves")
    src, so = d / "shim.cpp", d / "shim.so"
    src.write_text(SHIM)
    fd.lib()
    subprocess.run(["g++", "-std=c++17", "-O1", "-w", "-fPIC", "-shared", "-D__HIP_PLATFORM_AMD__", f"-I{root}",
                    "-I/opt/rocm/include", str(src), "-o", str(so), fd.LIB_PATH,
                    f"-Wl,-rpath,{os.path.dirname(fd.LIB_PATH)}", "-Wl,--unresolved-symbols=ignore-in-shared-libs"],
                   check=True)
    return ctypes.CDLL(str(so))


@pytest.mark.parametrize("w,h,narrow,wide", [(1, 1, 8, 8), (704, 704, 8, 8), (720, 720, 4, 8), (960, 960, 4, 8),
                                             (1348, 1348, 4, 8), (1360, 1360, 4, 4), (1920, 1080, 4, 4)])
def test_frames(shim, w, h, narrow, wide):
    """64-bit rows keep 8 waves on frames where 4 leave the longest lists to
    too few of them (soup of 1 M triangles, 720 x 720 receivers, 48 x 48
    samples: 1252 us with 4, 817 with 8)."""
    at = importlib.import_module("4dzb_amd.autotune")
    for res in (8, 32, 33, 64):
        want = wide if res > 32 else narrow
        assert shim.waves(w, h, res, 4) == want
        assert at.library_waves(res, w, h) == want
