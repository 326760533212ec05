"""The row loop's decisions (a limit by reciprocal and rounding, the sign of the
edges' least largest value) against the general form that follows the
reference's expressions, on random and adversarial edge planes (MI355X only):
what is decided without a division is the general form's mask, and the exact
form agrees everywhere."""
import numpy as np
import pytest

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
    for k, what in ((1, "decided"), (2, "exact")):
        bad = np.nonzero(out[:, k])[0]
        assert len(bad) == 0, (what, len(bad), [(coef[i].tolist(), hex(int(out[i, k]))) for i in bad[:3]])
    rows = sum(int(x).bit_count() if hasattr(int, "bit_count") else bin(int(x)).count("1") for x in out[:, 0])
    assert rows > 0.4 * R * len(coef)
