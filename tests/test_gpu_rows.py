"""The row loop's decisions (a limit by reciprocal and rounding, the sign of the
edges' least largest value) against the general form that follows the
reference's expressions, on random and adversarial edge planes (MI355X only):
what is decided without a division is the general form's mask, the exact form
agrees everywhere, and no row with a sample is outside the loop's row range.
Triangles that reach past the light's columns are not walked row by row between
their vertices."""
import numpy as np
import pytest

from parity import compare, failures
from test_gpu_rowwindow import _cases, _triangle_edges

pytestmark = pytest.mark.gpu


def _near(rng, R, n=60_000):
    out = []
    # edges through whole columns: small integers, and a few ulps beside them
    t = rng.integers(-8, 9, (n, 3, 3)).astype(np.float64)
    t[:, :, 2] = -(t[:, :, 0] * rng.integers(0, R + 1, (n, 3)) + t[:, :, 1] * rng.integers(-2, R + 3, (n, 3)))
    out.append(t)
    u = t.astype(np.float32)
    u = (u * (1 + rng.integers(-4, 5, u.shape).astype(np.float32) * np.float32(2.0 ** -23))).astype(np.float32)
    u *= (2.0 ** rng.integers(-40, 41, (n, 3, 1))).astype(np.float32)
    out.append(u)
    # limits within 2^-15 of a whole column, either side
    v = _triangle_edges(rng, n, R)
    r, c = rng.integers(0, R, (n, 3)), rng.integers(0, R + 1, (n, 3))
    v[:, :, 2] = -(v[:, :, 0] * r + v[:, :, 1] * (c + rng.choice([-1, 1], (n, 3)) * 2.0 ** rng.uniform(-24, -10, (n, 3))))
    out.append(v)
    # nearly parallel to the rows: limits millions of columns off, of every sign
    w = _triangle_edges(rng, n, R)
    w[:, :, 1] *= 10.0 ** rng.uniform(-12, -3, (n, 3))
    out.append(w)
    x = _triangle_edges(rng, n, R)
    i = rng.integers(0, 3, n)
    x[np.arange(n), i, 1] = rng.choice([0.0, -0.0, 1e-45, -1e-40, 1e-30, -1e-9], n)
    out.append(x)
    # the least largest value near zero at some row
    y = _triangle_edges(rng, n, R)
    k = rng.integers(0, 3, n)
    a, b = y[np.arange(n), k, 0], y[np.arange(n), k, 1]
    y[np.arange(n), k, 2] = -(a * rng.integers(0, R, n) + np.maximum(b * (R - 1), 0)) * (1 + rng.integers(-30, 31, n) * 2.0 ** -23)
    out.append(y)
    return np.concatenate(out).astype(np.float32).reshape(-1, 9)


@pytest.mark.parametrize("R", [1, 2, 7, 8, 16, 31, 32, 33, 63, 64])
def test_rows_decided_as_by_the_general_form(fd, R):
    rng = np.random.default_rng(300 + R)
    coef = np.concatenate([_cases(rng, R), _near(rng, R)])
    print(f"[rows] R={R} triples={len(coef)}", flush=True)
    out = fd.selftest_rows(coef, R)
    for k, what in ((1, "decided"), (2, "exact"), (3, "left out")):
        bad = np.nonzero(out[:, k])[0]
        assert len(bad) == 0, (what, len(bad), [(coef[i].tolist(), hex(int(out[i, k]))) for i in bad[:3]])
    rows = sum(int(x).bit_count() if hasattr(int, "bit_count") else bin(int(x)).count("1") for x in out[:, 0])
    assert rows > 0.4 * R * len(coef)


@pytest.mark.parametrize("pose", ["axial", "tilt"])
@pytest.mark.parametrize("res", [32, 64])
def test_long_triangles_visit_the_references_rows(fd, oracle, wl, res, pose):
    """Slivers many times the light's size, at 30 to 60 degrees to its rows.  The
    reference visits the rows of every edge's own range that are not full; the
    kernel those too, and where a pair's window spans at most 6 rows all of them:
    6 rows a pair more at the most."""
    rng = np.random.default_rng(res)
    n = 800
    c = np.stack([rng.uniform(-3, 3, n), rng.uniform(-3, 3, n), rng.uniform(1.0, 3.0, n)], 1)
    a = np.radians(rng.uniform(30, 60, n)) * rng.choice([-1, 1], n)
    d = np.stack([np.cos(a), np.sin(a), 0 * a], 1)
    nrm = np.stack([-np.sin(a), np.cos(a), 0 * a], 1)
    v = np.stack([c - 2.5 * d, c + 2.5 * d, c + 0.02 * nrm], 1).astype(np.float32)
    verts = np.ones((3 * n, 4), np.float32)
    verts[:, :3] = v.reshape(-1, 3)
    light = wl.LightDesc(0.25, 0.25, (0.1, -0.2, 4.0), res_w=res, res_h=res)
    if pose == "tilt":
        light.view_dir, light.up_dir = (0.1, -0.05, -1.0), (0.1, 1.0, 0.0)
    frame = wl.Frame(f"slivers-{res}-{pose}", wl.Scene(verts, np.arange(3 * n, dtype=np.int32).reshape(-1, 3)),
                     wl.receivers_plane(48, 40, 4.0), light, backface_cull=0)
    print(f"[rows] {frame.name}", flush=True)
    rep, fr, o = compare(fd, oracle, frame, stages=False)
    assert o.exit == 0 and not failures(rep), failures(rep)
    fr.ctx.set_profiling(False, True)
    rc, _ = fr.run()
    _, ops = fr.ctx.get_profile(ops=True)
    fr.close()
    assert rc == 0 and ops[6] > 100_000
    assert ops[2] <= ops[6] + 6 * ops[7], ops
