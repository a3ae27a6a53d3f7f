"""The inverse Cholesky factor with dropped columns (panels of 16 columns,
32 x 32 tiles) inside derek_hip_hegv, against numpy on the kept columns.

Sizes on both sides of panel and tile edges; dependent and zero columns at
the first, last and inner positions of a panel, several in one panel, a whole
panel.  The overlap of the kept columns has a condition number below 20, so
eigenvalues and residuals of an m x m problem hold to a few m * cond * eps *
|H|: below 3e-12 * |H| at m = 640 (eps 1.1e-16).
"""
import numpy as np
import pytest

from derek_amd import lib

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = lib.Context((8, 8, 8), 1, 4, 1.0, 1)
    yield c
    c.close()


CASES = [(1, []), (2, [1]), (15, []), (16, [15]), (17, [0]), (17, [16]), (31, [3, 15, 16]), (32, []), (33, [32]),
         (47, list(range(16, 32))), (48, [2, 3, 4, 30]), (49, [48]), (64, [17, 47]), (80, []), (113, [16, 31, 32, 111]),
         (160, [100, 159]), (300, [5, 64, 250]), (600, [16, 299]), (640, [])]


@pytest.mark.parametrize("m,dead", CASES)
def test_hegv_dropped_columns(ctx, m, dead):
    print("hegv chol", m, dead, flush=True)
    rng = np.random.default_rng(m + len(dead))
    n = 3 * m + 8
    y = (rng.normal(size=(n, m)) + 1j * rng.normal(size=(n, m))) * rng.uniform(0.3, 3.0, m)
    for i, j in enumerate(dead):
        # a zero column, or a multiple of an earlier kept one
        kept = [q for q in range(j) if q not in dead]
        y[:, j] = y[:, kept[(3 * i) % len(kept)]] * (1.7 - 0.4j) if kept and i % 2 == 0 else 0.0
    d = rng.uniform(-1.0, 4.0, n)
    S, H = y.conj().T @ y, y.conj().T @ (d[:, None] * y)
    keep = [q for q in range(m) if q not in dead]
    nev = max(1, len(keep) // 2)
    w, c = ctx.hegv(S, H, nev)
    s, h = S[np.ix_(keep, keep)], H[np.ix_(keep, keep)]
    li = np.linalg.inv(np.linalg.cholesky(s))
    ref = np.linalg.eigvalsh(li @ h @ li.conj().T)[:nev]
    assert np.all(c[dead] == 0)
    assert np.max(np.abs(w - ref)) < 3e-12 * 4.0
    ck = c[keep]
    assert np.max(np.abs(ck.conj().T @ s @ ck - np.eye(nev))) < 3e-12
    scale = np.abs(s).max()
    assert np.max(np.abs(h @ ck - s @ ck * w)) < 3e-12 * 4.0 * np.sqrt(scale) * 10.0
