"""The occlusion's projected sample window and its block prefilter, bit-exact
against the oracle where their bounds are tight or do not hold (MI355X only):
slivers and edge-on triangles (the window's margin), vertices below the
receivers or above the light, huge and tiny triangles (no window), edges along
the light axes with coordinates on the sample grid (quotients that are whole
numbers, planes with zero coefficients), lights along the axes, tilted, and
facing up, and the sizes at the edges of the row words and column strips."""
import numpy as np
import pytest

from parity import compare, failures

pytestmark = pytest.mark.gpu


def _tris(kind, n, rng):
    c = np.stack([rng.uniform(-3, 3, n), rng.uniform(-3, 3, n), rng.uniform(0.4, 3.0, n)], 1)
    e = rng.normal(size=(n, 3, 3)) * 0.25
    if kind == "sliver":      # almost collinear vertices
        d = rng.normal(size=(n, 1, 3))
        e = d * np.array([0.0, 0.5, 1.0])[None, :, None] + rng.normal(size=(n, 3, 3)) * 10.0 ** rng.uniform(-6, -2, (n, 1, 1))
    elif kind == "edge_on":   # vertical triangles: seen from the side by the receivers below
        a = rng.uniform(0, 2 * np.pi, n)
        u = np.stack([np.cos(a), np.sin(a), 0 * a], 1)[:, None, :]
        e = u * rng.normal(size=(n, 3, 1)) * 0.5 + np.array([0, 0, 1.0]) * rng.normal(size=(n, 3, 1)) * 0.3
    elif kind == "straddle":  # vertices below the receivers, others above the light
        c[:, 2] = np.where(rng.random(n) < 0.7, 0.05, 3.9)
        e = rng.normal(size=(n, 3, 3)) * np.array([0.5, 0.5, 0.4])
    elif kind == "scales":    # edges from 1e-4 to 1, and two huge triangles over x > 2.6, x < -3.1
        e *= 10.0 ** rng.uniform(-3.5, 0.2, (n, 1, 1))
        e[:, :, 2] = np.clip(e[:, :, 2], -0.3, 0.3)
        c[:2] = 0.0
        e[0] = [[2.6, -700, 1.5], [2.6, 500, 1.7], [9000, 3, 1.6]]
        e[1] = [[-3.1, 600, 2.0], [-3.1, -500, 2.0], [-800, -7, 2.2]]
    elif kind == "grid":      # corners of a coarse grid: exact ties and zero coefficients
        c = np.round(c * 4) / 4
        e = np.round(e * 6) / 8
    return c[:, None, :] + e


def _frame(wl, kinds, res, pose, cull, seed, n=400, w=52, h=45, offset=(0.0, 0.0, 0.0)):
    rng = np.random.default_rng(seed)
    v = np.concatenate([_tris(k, n, rng) for k in kinds])
    flip = pose == "up"
    xy = np.stack(np.meshgrid(np.linspace(-4, 4, w), np.linspace(-4, 4, h)), -1)
    pos = np.ones((h, w, 4), np.float32)
    pos[..., :2] = xy
    pos[..., 2] = 0.1 * np.sin(3 * xy[..., 0]) * np.cos(2 * xy[..., 1]) if "grid" not in kinds else 0.0
    nrm = np.zeros((h, w, 4), np.float32)
    nrm[..., 2] = 1.0
    light = wl.LightDesc(0.75, 0.5, (0.25, -0.5, 4.0), res_w=res, res_h=res)
    if pose == "tilt":
        light.view_dir, light.up_dir = (0.25, -0.15, -1.0), (0.2, 1.0, 0.1)
    if flip:   # the scene upside down: the light below, facing up
        v[..., 2] *= -1
        pos[..., 2] *= -1
        nrm[..., 2] *= -1
        light.position, light.view_dir = (0.25, -0.5, -4.0), (0.0, 0.0, 1.0)
    off = np.asarray(offset)
    v = v + off
    pos[..., :3] += off.astype(np.float32)
    light.position = tuple(float(a) for a in np.asarray(light.position) + off)
    verts = np.ones((3 * len(v), 4), np.float32)
    verts[:, :3] = v.reshape(-1, 3)
    scene = wl.Scene(verts, np.arange(3 * len(v), dtype=np.int32).reshape(-1, 3))
    return wl.Frame(f"{'+'.join(kinds)}-{pose}-r{res}", scene, wl.Receivers(pos, nrm), light, backface_cull=cull)


KINDS = ["sliver", "edge_on", "straddle", "scales", "grid"]


def _check(fd, oracle, frame):
    print(f"[window] {frame.name} cull {frame.backface_cull}", flush=True)
    rep, fr, o = compare(fd, oracle, frame)
    fr.close()
    assert o.exit == 0 and int(o.scalars["pairs"]) > 0
    assert not failures(rep), failures(rep)


@pytest.mark.parametrize("pose", ["axial", "tilt", "up"])
@pytest.mark.parametrize("kind", KINDS)
def test_window_kinds(fd, oracle, wl, kind, pose):
    _check(fd, oracle, _frame(wl, [kind], 24 if pose != "tilt" else 40, pose, 0, seed=11, n=200))


@pytest.mark.parametrize("res", [1, 2, 5, 8, 9, 16, 17, 31, 32, 33, 63, 64])
def test_window_grid_sizes(fd, oracle, wl, res):
    _check(fd, oracle, _frame(wl, KINDS, res, "axial", 1, seed=100 + res, n=40))


@pytest.mark.parametrize("res", [16, 64])
def test_window_far_from_origin(fd, oracle, wl, res):
    _check(fd, oracle, _frame(wl, ["sliver", "edge_on"], res, "axial", 0, seed=7, offset=(300.0, -200.0, 50.0)))


@pytest.mark.parametrize("res", [32, 64])
def test_window_dense_occupancy(fd, oracle, wl, res):
    """Long lists over few receivers: most triangles meet full rows (strips)."""
    _check(fd, oracle, _frame(wl, ["scales", "edge_on", "sliver"], res, "axial", 0, seed=5, n=2500, w=24, h=16))
