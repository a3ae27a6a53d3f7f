"""Eigenpairs at the edges of the one-workgroup tridiagonalisation: its 16 x 16
register tiles, the wavefront that forms the reflectors (an idle one up to 112
columns), and the 128 columns from which on multi-workgroup steps come first.

Bounds: Householder reduction, bisection and inverse iteration are backward
stable, with errors of a few n eps |A|; the bounds are those of the other
eigenvalue tests (1e-12 n for the values, 1e-11 sqrt(n) for residual and
orthogonality, relative to the largest eigenvalue).
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


def check(ctx, A):
    n = len(A)
    w, Z = ctx.heev(A, n)
    ref = np.linalg.eigvalsh(A)
    scale = max(np.abs(ref).max(), 1e-300)
    assert np.max(np.abs(w - ref)) < 1e-12 * scale * n
    assert np.max(np.abs(A @ Z - Z * w[None, :])) < 1e-11 * scale * np.sqrt(n)
    assert np.max(np.abs(Z.conj().T @ Z - np.eye(n))) < 1e-11 * np.sqrt(n)


@pytest.mark.parametrize("n", [4, 15, 18, 31, 32, 47, 48, 49, 63, 65, 66, 95, 111, 113, 126, 127, 129, 130, 131, 145])
def test_tile_edges(ctx, n):
    print("tridiag", n, flush=True)
    rng = np.random.default_rng(n)
    A = rng.normal(size=(n, n)) + 1j * rng.normal(size=(n, n))
    A = A + A.conj().T
    check(ctx, A)
    check(ctx, 1e-30 * A)
    # a diagonal block at the end and one dense corner: columns without a
    # reflector before and after ones with
    k = n // 3
    A[k:, :] = A[:, k:] = 0
    A[np.arange(k, n), np.arange(k, n)] = np.arange(k, n)
    A[n - 1, 0] = A[0, n - 1] = 0.5
    check(ctx, A)


@pytest.mark.parametrize("n,seed", [(18, 3), (47, 0), (65, 6), (95, 5)])
def test_rows_decoupled_from_the_rest(ctx, n, seed):
    """A diagonal row whose eigenvalue is met to the last bit: the shifted
    matrix then has an exactly zero pivot."""
    rng = np.random.default_rng(n + 1000 * seed)
    A = rng.normal(size=(n, n)) + 1j * rng.normal(size=(n, n))
    A = A + A.conj().T
    k = n // 3
    A[k:, :] = A[:, k:] = 0
    A[np.arange(k, n), np.arange(k, n)] = np.arange(k, n)
    A[n - 1, 0] = A[0, n - 1] = 0.5
    check(ctx, A)


@pytest.mark.parametrize("n", [192, 256, 257, 258, 320, 448, 449, 450, 577, 640, 641, 642, 700])
def test_multi_workgroup_steps(ctx, n):
    """Trailing rows at the edges of the register steps (256, 448 and 640 rows)
    and beyond them; columns without a reflector among the others."""
    print("wide steps", n, flush=True)
    rng = np.random.default_rng(n)
    A = rng.normal(size=(n, n)) + 1j * rng.normal(size=(n, n))
    A = A + A.conj().T
    for q in (1, 2, n - 200, n - 130):
        if q > 0:  # column q - 1 keeps its diagonal and sub-diagonal only
            A[q + 1:, :q] = 0
            A[:q, q + 1:] = 0
    check(ctx, A)
