"""The counting sorts' kernels at the edges of their blocks, every stage
bit-exact against the oracle (MI355X only): receiver and triangle counts around
a wave (64), a block (1024) and a scan block (4096), all grids, triangles that
cover from one bin to the whole light plane, frames with receivers but without
pairs."""
import numpy as np
import pytest

from parity import compare, failures

pytestmark = pytest.mark.gpu


def _frame(wl, w, h, ntris, grid_log2, seed, above=True):
    rng = np.random.default_rng(seed)
    c = np.stack([rng.uniform(-3, 3, ntris), rng.uniform(-3, 3, ntris), rng.uniform(0.4, 3.0, ntris)], 1)
    size = 10.0 ** rng.uniform(-2, -0.7, (ntris, 1, 1))
    size[::97] = 6.0   # the whole light plane
    v = c[:, None, :] + rng.normal(size=(ntris, 3, 3)) * size * np.array([1.0, 1.0, 0.05])
    if not above:
        v[..., 2] = -3.0 - 0.01 * v[..., 2]   # below the receivers: no bin test passes
    verts = np.ones((3 * ntris, 4), np.float32)
    verts[:, :3] = v.reshape(-1, 3)
    scene = wl.Scene(verts, np.arange(3 * ntris, dtype=np.int32).reshape(-1, 3))
    pos = np.ones((h, w, 4), np.float32)
    pos[..., :2] = rng.uniform(-4, 4, (h, w, 2))   # neighbours in different bins
    pos[..., 2] = rng.uniform(0, 0.2, (h, w))
    pos[rng.random((h, w)) < 0.05] = np.nan
    pos[0, 0] = (0.0, 0.0, 0.1, 1.0)
    nrm = np.zeros((h, w, 4), np.float32)
    nrm[..., 2] = np.where(rng.random((h, w)) < 0.1, -1.0, 1.0)
    nrm[0, 0, 2] = 1.0
    return wl.Frame(f"{w}x{h}-t{ntris}-g{grid_log2}", scene, wl.Receivers(pos, nrm),
                    wl.LightDesc(0.75, 0.5, (0.25, -0.5, 4.0), res_w=4, res_h=4), backface_cull=0, grid_log2=grid_log2)


SIZES = [(1, 1, 1), (8, 8, 63), (9, 8, 65), (32, 32, 1023), (33, 32, 1024), (128, 32, 1025), (129, 33, 4095), (64, 65, 4097)]


@pytest.mark.parametrize("grid_log2", [3, 4, 5, 6])
@pytest.mark.parametrize("w,h,ntris", SIZES)
def test_sort_edges(fd, oracle, wl, w, h, ntris, grid_log2):
    frame = _frame(wl, w, h, ntris, grid_log2, seed=w * h + ntris + grid_log2)
    print(f"[sort] {frame.name}", flush=True)
    rep, fr, o = compare(fd, oracle, frame)
    fr.close()
    assert not failures(rep), (o.exit, failures(rep))
    if w * h >= 1024:
        assert o.exit == 0


@pytest.mark.parametrize("grid_log2", [3, 6])
def test_sort_without_pairs(fd, oracle, wl, grid_log2):
    frame = _frame(wl, 65, 40, 500, grid_log2, seed=3, above=False)
    print(f"[sort] no pairs {frame.name}", flush=True)
    rep, fr, o = compare(fd, oracle, frame)
    fr.close()
    assert o.exit != 0 and not failures(rep), (o.exit, failures(rep))
