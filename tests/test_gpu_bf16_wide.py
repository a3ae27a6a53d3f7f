"""The two-term BF16 products on 128-column tiles: overlaps (over 64
columns on both sides and 131072 rows) and rotations with at least one 128-row
workgroup per CU, at ragged sizes, against the exact product of the complex64
operands.

A two-term product keeps about 16 bits: the repository's two-term bound, 1e-4
of the largest value.
"""
import numpy as np
import pytest

from derek_amd import lib
from tests.conftest import assert_close

pytestmark = pytest.mark.gpu


def block(rng, m, npw):
    return (rng.normal(size=(m, npw)) + 1j * rng.normal(size=(m, npw))).astype(np.complex64)


def check(got, a, b, sign, what):
    """a^T b of complex64 columns a (k, i), b (k, j); sign -1 conjugates a."""
    a, b = a.astype(complex), b.astype(complex)
    assert_close(got, (a.conj() if sign < 0 else a).T @ b, 1e-4, what)


@pytest.mark.parametrize("npw,m,n", [(131073, 65, 129), (131072, 128, 66), (140015, 129, 129), (133007, 70, 70)])
def test_wide_overlap(npw, m, n):
    print("wide overlap", npw, m, n, flush=True)
    rng = np.random.default_rng(npw)
    ctx = lib.Context((8, 8, 8), 1, 1, 1.0, 1, lib.DEREK_MIXED)
    x, y = block(rng, m, npw), block(rng, n, npw)
    check(ctx.overlap(x, y), x.T, y.T, -1, f"{m}x{n}")
    if m == n:
        s = ctx.overlap(x, x)
        check(s, x.T, x.T, -1, f"{m} Hermitian")
        assert np.array_equal(s, s.conj().T)
    ctx.close()


@pytest.mark.parametrize("npw", [32769, 40000, 65535])
def test_wide_rotation(npw):
    rng = np.random.default_rng(npw)
    ctx = lib.Context((8, 8, 8), 1, 1, 1.0, 1, lib.DEREK_MIXED)
    for m, n in [(1, 1), (15, 16), (17, 33), (48, 24), (33, 129), (130, 70)]:
        print("wide rotation", npw, m, n, flush=True)
        x, u = block(rng, m, npw), block(rng, m, n)
        got = ctx.rotate(x, u)
        check(got, u, x, 1, f"{m}->{n}")
    ctx.close()
