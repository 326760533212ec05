"""The application stages at the largest tables that travel in a launch's
arguments and the first ones that are uploaded (MI355X only)."""
import numpy as np
import pytest

from test_gpu_app import SHADE_ATOL, SHADE_RTOL

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nbox", [0, 1, 40, 41])
def test_gbuffer_box_tables(fd, wl, nbox):
    print(f"[tables] {nbox} boxes", flush=True)
    sc = wl.gbuffer_scene_boxes(131, 77, nbox, 9)
    ref = wl.gbuffer_boxes_host(sc)
    for targets in (2, 4):
        g = [fd.DeviceBuffer(131 * 77 * 16) for _ in range(targets)]
        strm = fd.Stream()
        fd.gbuffer_boxes(131, 77, sc.boxes, sc.materials if targets == 4 else None, sc.eye, sc.at, sc.up, sc.fovy_deg,
                         sc.ground_half, *g, stream=strm)
        strm.sync()
        strm.close()
        for k in range(targets):
            got = g[k].download(np.float32).reshape(77, 131, 4)
            want = ref[k].copy()
            if targets == 2:   # no materials: w is 1 on a hit
                want[..., 3] = np.where(np.isnan(ref[0][..., 0]), want[..., 3], 1.0)
            same = (got.view(np.uint32) == want.view(np.uint32)) | (np.isnan(got) & np.isnan(want))
            assert same.all(), (nbox, targets, k, int((~same).sum()))


@pytest.mark.parametrize("ns", [1, 320, 321])
def test_shade_sample_tables(fd, wl, oracle, ns):
    print(f"[tables] {ns} samples", flush=True)
    w, h = 61, 37
    r = np.random.default_rng(ns)
    sc = wl.gbuffer_scene_boxes(w, h, 6, 4)
    host = wl.gbuffer_boxes_host(sc)
    g = [fd.DeviceBuffer.from_array(np.ascontiguousarray(x, np.float32)) for x in host]
    sh = r.uniform(0, 1, w * h).astype(np.float32)
    shadow = fd.DeviceBuffer.from_array(sh)
    samples = [np.array([r.uniform(-2, 2), r.uniform(-2, 2), 6.0]) for _ in range(ns)]
    La, Ld, Ls = (0.2, 0.2, 0.2), (0.9, 0.85, 0.8), (0.5, 0.5, 0.5)
    rgba = fd.DeviceBuffer(w * h * 16)
    strm = fd.Stream()
    fd.shade(w, h, samples, sc.eye, La, Ld, Ls, shadow, *g, rgba, stream=strm)
    strm.sync()
    strm.close()
    got = rgba.download(np.float32).reshape(-1, 4)
    want = oracle.shade(sh, *[np.asarray(x, np.float32).reshape(-1, 4) for x in host], samples, sc.eye, La, Ld, Ls)
    assert np.array_equal(np.isnan(got), np.isnan(want))
    ok = ~np.isnan(want)
    # one sample's tolerance, and one rounding more per term of the sum
    assert ok.any() and np.allclose(got[ok], want[ok], rtol=SHADE_RTOL + ns * 2.0 ** -24, atol=SHADE_ATOL)
