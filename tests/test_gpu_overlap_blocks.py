"""Overlaps whose 64 x 64 tiles hold every number of needed 16 x 16 blocks
(1 to 16, Hermitian diagonal tiles and general ones), so that every split of
blocks and slab rows over the wavefronts runs, against the oracle; short,
ragged and single row chunks.

A sum of npw products carries at most npw * eps of the sum of their moduli,
in practice sqrt(npw) * eps: 1e-13 (FP64) and 1e-5 (FP32 matrix cores) of the
largest value, as in the other overlap tests.
"""
import numpy as np
import pytest

from derek_amd import lib
from oracle import ks as oks
from tests.conftest import assert_close

pytestmark = pytest.mark.gpu

SHAPES = [(1, 1), (10, 10), (16, 17), (20, 20), (24, 24), (33, 33), (33, 20), (48, 48), (49, 49), (40, 60), (64, 64),
          (64, 10), (50, 49), (65, 65), (80, 80), (113, 70), (160, 160), (7, 130)]


@pytest.mark.parametrize("precision", [lib.DEREK_FP64, lib.DEREK_MIXED])
@pytest.mark.parametrize("npw", [1, 37, 1503, 4099])
def test_overlap_block_splits(precision, npw):
    rng = np.random.default_rng(npw)
    ctx = lib.Context((8, 8, 8), 1, 4, 1.0, 1, precision)
    if precision == lib.DEREK_MIXED:
        ctx.set_gemm(0)
    tol = 1e-13 if precision == lib.DEREK_FP64 else 1e-5
    for m, n in SHAPES:
        print("overlap blocks", precision, npw, m, n, flush=True)
        x = rng.normal(size=(m, npw)) + 1j * rng.normal(size=(m, npw))
        y = rng.normal(size=(n, npw)) + 1j * rng.normal(size=(n, npw))
        assert_close(ctx.overlap(x, y), oks.overlap(x, y), tol, f"{m}x{n}")
        if m == n:
            assert_close(ctx.overlap(x, x), oks.overlap(x, x), tol, f"{m}x{n} Hermitian")
    ctx.close()
