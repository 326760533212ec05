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
    return fd_default_waves(res, a.chunkSlots);
}
// instances per occlusion class (32 / 64-bit rows x 2 / 4 / 8 waves) of a batch of n frames
extern "C" void batch(int n, int w, int h, int res, int asked, int* classes) {
    std::vector<FdArgs> args(n);
    const fdh::Model md{nullptr, 4, 3, nullptr, 1};
    FdLight L{};
    L.res = res;
    L.wpr = res > 32 ? 2 : 1;
    for (FdArgs& a : args) {
        fdh::fill_args(a, md, nullptr, nullptr, w, h, L, 0.0f, 0, 4, 3, nullptr, nullptr, 1);
        a.wavesReq = asked;
        a.occWaves = asked ? asked : fd_default_waves(L.res, a.chunkSlots);
    }
    std::vector<char> image;
    FdBatchPlan P;
    fdh::build_plan(args, true, nullptr, image, P);
    for (int c = 0; c < FD_OCC_CLASSES; ++c) classes[c] = P.nocc[c];
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


@pytest.mark.parametrize("w,h,narrow,wide,widest", [
    (1, 1, 8, 8, 8), (704, 704, 8, 8, 8), (720, 720, 4, 8, 8), (960, 960, 4, 8, 8), (1348, 1348, 4, 8, 8),
    (1360, 1360, 4, 4, 8), (1920, 1080, 4, 4, 8), (1692, 1692, 4, 4, 8), (1700, 1700, 4, 4, 4), (2560, 1440, 4, 4, 4)])
def test_frames(shim, w, h, narrow, wide, widest):
    """64-bit rows keep 8 waves on frames where 4 leave the longest lists to
    too few of them (soup of 1 M triangles, 720 x 720 receivers, 48 x 48
    samples: 1252 us with 4, 817 with 8), and above 48 x 48 samples, where LDS
    holds 4 work items of 4 waves per CU, on larger ones (tessellated boxes of
    1.2 M triangles that the receivers lie on, 1920 x 1080, 64 x 64: 7602, 5949)."""
    at = importlib.import_module("4dzb_amd.autotune")
    for res in (8, 32, 33, 48, 49, 64):
        want = widest if res > 48 else wide if res > 32 else narrow
        assert shim.waves(w, h, res, 4) == want
        assert at.library_waves(res, w, h) == want


@pytest.mark.parametrize("n,w,h,res,asked,waves", [
    (2, 512, 512, 8, 0, 8), (16, 256, 256, 32, 0, 8),      # 8706 and 20496 work items: too few to fill the GPU with 4
    (6, 512, 512, 16, 0, 8), (22, 256, 256, 16, 0, 8),     # 26118, 28182
    (23, 256, 256, 16, 0, 4), (8, 512, 512, 32, 0, 4),     # 29463, 34824
    (26, 256, 256, 64, 0, 8), (300, 256, 256, 33, 0, 8),   # 64-bit rows: by the frame
    (2, 1920, 1080, 48, 0, 4), (2, 1920, 1080, 64, 0, 8), (2, 720, 720, 16, 0, 4), (26, 256, 256, 16, 2, 2), (26, 256, 256, 16, 8, 8)])
def test_batches(shim, n, w, h, res, asked, waves):
    """Small frames of 32-bit rows take 4 waves in batches that fill the GPU
    with that (soup of 300 k triangles, two 512 x 512 frames with 8 x 8
    samples: 800 us with 4, 608 with 8); an asked count stays."""
    got = (ctypes.c_int * 6)()
    shim.batch(n, w, h, res, asked, got)
    want = [0] * 6
    want[(3 if res > 32 else 0) + {2: 0, 4: 1, 8: 2}[waves]] = n
    assert list(got) == want


def test_untuned_classes_take_the_librarys_default():
    """Where no count was tuned the tables ask for none, and the layouts name
    the library's own (a large frame of 64-bit rows: 4)."""
    at = importlib.import_module("4dzb_amd.autotune")
    assert at.default_layout(64, 2560, 1440) == (16, 8, 4) and at.default_layout(64, 1024, 1024) == (16, 8, 8)
    assert at.default_layout(64, 2560, 1440) in at.CANDIDATES
    cache = {at.class_key(0, 2560, 1440, 64): dict(bins=16, tile=8, ms=1.0, default_ms=1.0, candidates={}),
             at.class_key(0, 256, 256, 16): dict(bins=16, tile=8, waves=4, ms=1.0, default_ms=1.0, candidates={})}
    assert at.layout(cache, 0, 2560, 1440, 64) == (16, 8, 4) and at.layout({}, 0, 2560, 1440, 64) == (16, 8, 4)
    assert at.layout(cache, 0, 256, 256, 16) == (16, 8, 4)
    assert sorted((t["w"], t["waves"]) for t in at.server_table(cache)) == [(256, 4), (2560, 0)]
