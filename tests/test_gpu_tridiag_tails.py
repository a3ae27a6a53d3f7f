"""Eigenpairs of matrices whose columns are almost reduced: a tridiagonal matrix
of O(1) plus a dense part so small that a column's entries below the
sub-diagonal vanish beside it when squared and added (their sum of squares, 4e-17, is
below half an ulp of the sub-diagonal's), but not in the spectrum's bounds.  Every step
of the reduction meets such a column: in registers, several workgroups wide (up
to 640 rows) and beyond.

Bounds: those of the other eigenvalue tests.  Dropping the small part would
leave a residual of up to its norm, about 1e-8: nine times the bound at n = 700.
"""
import numpy as np
import pytest

from derek_amd import lib
from tests.test_gpu_tridiag import check

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [3, 60, 128, 129, 200, 640, 700])
def test_small_entries_below_the_sub_diagonal(n):
    print("tridiag tails", n, flush=True)
    rng = np.random.default_rng(n)
    g = (rng.normal(size=(n, n)) + 1j * rng.normal(size=(n, n))) * (3e-9 / np.sqrt(n))
    A = g + g.conj().T
    i = np.arange(n)
    A[i, i] = rng.uniform(-1.0, 3.0, n)
    sub = rng.uniform(0.8, 1.2, n - 1) * np.exp(2j * np.pi * rng.uniform(size=n - 1))
    A[i[1:], i[:-1]] = sub
    A[i[:-1], i[1:]] = sub.conj()
    # the same with one column of that kind before dense ones
    B = rng.normal(size=(n, n)) + 1j * rng.normal(size=(n, n))
    B = B + B.conj().T
    B[1:, 0], B[0, 1:] = A[1:, 0], A[0, 1:]
    ctx = lib.Context((8, 8, 8), 1, 4, 1.0, 1)
    check(ctx, A)
    check(ctx, B)
    ctx.close()
