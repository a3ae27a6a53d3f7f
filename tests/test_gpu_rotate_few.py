"""The two-term rotation on 128-row workgroups for at most 32 columns of X, which
takes it from 1024 workgroups on, on both sides of that number; against the
exact product of the complex64 operands, with the two-term bound of the other
tests, 1e-4 of the largest value.
"""
import numpy as np
import pytest

from derek_amd import lib
from tests.test_gpu_bf16_wide import block, check

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("npw", [130944, 130945, 131073, 140000])
@pytest.mark.parametrize("m,n", [(1, 1), (15, 16), (17, 33), (32, 16), (33, 16)])
def test_rotation_of_few_columns(npw, m, n):
    print("rotation of few columns", npw, m, n, flush=True)
    rng = np.random.default_rng(npw + m)
    ctx = lib.Context((8, 8, 8), 1, 1, 1.0, 1, lib.DEREK_MIXED)
    x, u = block(rng, m, npw), block(rng, m, n)
    check(ctx.rotate(x, u), u, x, 1, f"{m}->{n}")
    ctx.close()
