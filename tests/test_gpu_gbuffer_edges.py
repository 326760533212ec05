"""The G-buffer producer's single-precision box test where distances tie or it
must not decide, bit-identical to the host ray cast (MI355X only): boxes that
share faces and edges, flat and inverted boxes, corners that are not finite,
an eye inside a box and on its face, rays along the axes, views narrower or
lower than a tile, the largest box count."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _scene(wl, w, h, boxes, **kw):
    boxes = np.asarray(boxes, np.float64).reshape(-1, 6)
    return wl.GbufferScene(w, h, boxes, wl.boxes_materials(len(boxes)), **kw)


def _grid_boxes(n):
    """n x n unit boxes, faces and edges shared."""
    return [(x - n / 2, y - n / 2, 0, x + 1 - n / 2, y + 1 - n / 2, 1 + (x + y) % 2) for x in range(n) for y in range(n)]


INF, NAN = float("inf"), float("nan")
CASES = {
    "shared-faces": dict(w=161, h=97, boxes=_grid_boxes(6)),
    "limit-256": dict(w=80, h=50, boxes=_grid_boxes(16)),
    "flat": dict(w=97, h=64, boxes=[(-2, -2, 1, 2, 2, 1), (1, -3, 0, 1, 3, 2), (-3, 0, 0, 3, 0, 3), (0, 0, 0, 0, 0, 4)]),
    "inverted": dict(w=97, h=64, boxes=[(2, 2, 2, -2, -2, 0), (-4, 3, 0, -3, 1, 1.5), (3, -1, 2, 4, -2, 0)]),
    "not-finite": dict(w=97, h=64, boxes=[(NAN, -1, 0, 1, 1, 1), (-INF, 2, 0, INF, 3, 1), (2, 2, NAN, 3, 3, 2),
                                          (-3, -3, 0, -2, -2, INF), (-1e35, -5, 0, 1e35, -4.5, 0.5)]),
    "eye-inside": dict(w=64, h=64, boxes=[(-20, -20, -1, 20, 20, 30), (-1, -1, 0, 1, 1, 1)]),
    "eye-on-face": dict(w=64, h=64, boxes=[(-1, -13.0, 0, 1, -12, 9.0), (-1, -14, 9.0, 1, -12, 10), (0, -13.0, 9.0, 2, 0, 11)]),
    # an odd view centred on an axis: components of the middle rays are exact zeros
    "along-y": dict(w=65, h=65, boxes=_grid_boxes(4), eye=(0.0, -10.0, 0.5), at=(0.0, 0.0, 0.5)),
    "straight-down": dict(w=33, h=35, boxes=_grid_boxes(4), eye=(0.0, 0.0, 9.0), at=(0.0, 0.0, 0.0), up=(0.0, 1.0, 0.0)),
    "narrow": dict(w=15, h=300, boxes=_grid_boxes(3)),
    "one-column": dict(w=1, h=77, boxes=_grid_boxes(3)),
    "low": dict(w=300, h=15, boxes=_grid_boxes(3)),
    "one-tile": dict(w=16, h=16, boxes=_grid_boxes(3)),
    "tile-plus-one": dict(w=17, h=33, boxes=_grid_boxes(3)),
}


@pytest.mark.parametrize("name", sorted(CASES))
def test_gbuffer_edges(fd, wl, name):
    print(f"[gbuffer] {name}", flush=True)
    sc = _scene(wl, **CASES[name])
    ref = wl.gbuffer_boxes_host(sc)
    g = [fd.DeviceBuffer(sc.width * sc.height * 16) for _ in range(4)]
    fd.gbuffer_boxes(sc.width, sc.height, sc.boxes, sc.materials, sc.eye, sc.at, sc.up, sc.fovy_deg, sc.ground_half, *g)
    fd.lib().fd_device_sync()
    for k in range(4):
        got = g[k].download(np.float32).reshape(sc.height, sc.width, 4)
        # a NaN's payload is not part of the contract beyond the background's
        same = (got.view(np.uint32) == ref[k].view(np.uint32)) | (np.isnan(got) & np.isnan(ref[k]))
        assert same.all(), (name, f"target g{k}", int((~same).sum()))
    if name in ("shared-faces", "inverted", "eye-inside"):
        assert (ref[3][..., 0] > 0).any()
