"""The occlusion's windows for a whole work item and the pairs that rely on
them, bit-exact against the oracle (MI355X only): lists long enough for them
(2 waves per work item, 8 x 8 bins), receivers on one level and on several,
where the triangles lie above, between and below them, every kind of triangle
whose bounds are tight or do not hold, and an "on the triangle" distance that
some pairs are within."""
import numpy as np
import pytest

from parity import compare, failures
from test_gpu_window import KINDS, _frame

pytestmark = pytest.mark.gpu


def _levels(frame, kind, sign):
    """Receivers on steps (the light's side is +z for sign 1)."""
    pos = frame.rx.pos
    h, w = pos.shape[:2]
    y, x = np.mgrid[0:h, 0:w]
    if kind == "steps":
        z = np.where((x // 3 + y // 5) % 2 == 0, 0.0, 1.3)
    elif kind == "three":
        z = np.array([0.0, 0.4, 2.2])[(x // 2 + 2 * (y // 3)) % 3]
    else:
        z = 0.05 * np.sin(x) * np.cos(y)
    pos[..., 2] = sign * z.astype(np.float32)
    return frame


def _shrink(frame, f):
    """Triangles scaled about their centroids: sparse masks, rows that stay open."""
    v = frame.scene.verts[:, :3].reshape(-1, 3, 3)
    c = v.mean(axis=1, keepdims=True)
    v[:] = c + (v - c) * np.float32(f)


@pytest.mark.parametrize("levels", ["flat", "steps", "three"])
@pytest.mark.parametrize("pose", ["axial", "tilt", "up"])
@pytest.mark.parametrize("res", [7, 32, 40])
def test_tile_windows(fd, oracle, wl, res, pose, levels):
    frame = _frame(wl, KINDS, res, pose, 0, seed=res, n=1200, w=40, h=24)
    _shrink(frame, 0.2)
    frame = _levels(frame, levels, -1.0 if pose == "up" else 1.0)
    frame.grid_log2 = 3
    frame.eps = 1e-3 if levels != "three" else 0.3
    print(f"[tiles] {frame.name} {levels}", flush=True)
    frame.occ_waves, frame.list_split = 2, 1
    rep, fr, o = compare(fd, oracle, frame, stages=False)
    fr.close()
    assert o.exit == 0 and int(o.scalars["pairs"]) > 64 * 64   # lists of 64 entries and more
    assert not failures(rep), failures(rep)


@pytest.mark.parametrize("res", [16, 32, 64])
@pytest.mark.parametrize("split", [1, 4])
def test_nearly_parallel_edges(fd, oracle, wl, res, split):
    """Edges within a few units in the last place of the light's axes: their
    column limits lie millions of columns outside the grid.  split 4: lists too
    short for the work item's windows."""
    rng = np.random.default_rng(res)
    n = 6000
    p = np.stack([rng.uniform(-3, 3, n), rng.uniform(-3, 3, n), rng.uniform(0.4, 3.0, n)], 1).astype(np.float32)
    w, h = rng.uniform(0.05, 0.3, (2, n))
    v = np.repeat(p[:, None, :], 3, axis=1)
    along = rng.integers(0, 2, n)   # the axis of the first edge
    i = np.arange(n)
    v[i, 1, along] += w.astype(np.float32)
    v[i, 2, along] += (w * rng.uniform(0, 1, n)).astype(np.float32)
    v[i, 2, 1 - along] += h.astype(np.float32) * rng.choice([-1, 1], n).astype(np.float32)
    ulps = rng.integers(-3, 4, (n, 3, 3)).astype(np.float32)
    v = (v * (1 + ulps * np.float32(2.0 ** -23))).astype(np.float32)
    frame = _frame(wl, ["grid"], res, "axial", 0, seed=1, n=4, w=48, h=32)
    verts = np.ones((3 * n, 4), np.float32)
    verts[:, :3] = v.reshape(-1, 3)
    frame.scene = wl.Scene(verts, np.arange(3 * n, dtype=np.int32).reshape(-1, 3))
    frame.grid_log2, frame.occ_waves, frame.list_split = 3, 2, split
    print(f"[tiles] parallel r{res} split {split}", flush=True)
    rep, fr, o = compare(fd, oracle, frame, stages=False)
    fr.close()
    assert o.exit == 0 and not failures(rep), failures(rep)
