"""The C tile edge of the BF16 overlaps as a state of the context: a call that
sets something else, or gives back what get_tuning reports, leaves the large
two-term overlaps with their kernel, and an edge that the autotuner chose goes
when the number of terms does.  Same kernel, same order of operations: the
results are equal to the last bit.
"""
import numpy as np
import pytest

from derek_amd import config, lib
from derek_amd.scf import Setup

pytestmark = pytest.mark.gpu


def block():
    rng = np.random.default_rng(11)
    return (rng.normal(size=(72, 131072)) + 1j * rng.normal(size=(72, 131072))).astype(np.complex64)


def test_wide_overlap_keeps_its_kernel():
    x = block()
    ctx = lib.Context((8, 8, 8), 1, 1, 1.0, 1, lib.DEREK_MIXED)
    print("tile state", flush=True)
    ref = ctx.overlap(x, x)
    ctx.set_tiles(0, 2, 128)
    assert not np.array_equal(ctx.overlap(x, x), ref)  # another kernel
    ctx.set_tiles(0, 2, 0)
    assert np.array_equal(ctx.overlap(x, x), ref)
    ctx.set_tiles(z_sticks=32)
    assert np.array_equal(ctx.overlap(x, x), ref)
    t = ctx.tuning()
    ctx.set_tiles(t["z_sticks"], t["gemm_rounds"], t["gemm_tile"])
    assert np.array_equal(ctx.overlap(x, x), ref)
    assert ctx.tuning() == t
    ctx.close()


def test_autotuned_edge_goes_with_its_terms():
    x = block()
    ctx = lib.Context((8, 8, 8), 1, 1, 1.0, 1, lib.DEREK_MIXED)
    ref = ctx.overlap(x, x)
    ctx.close()
    spec = config.small_system(seed=3)
    ctx = Setup(spec).context(lib.DEREK_MIXED)
    for terms in (1, 3, 2):
        print("tile state, autotuned with", terms, flush=True)
        ctx.set_gemm(terms)
        ctx.scf_init(spec.nelec, kT=spec.kT, seed=spec.seed, autotune=True)
        t = ctx.tuning()
        assert t["gemm_tile"] in (64, 128)
        ctx.set_gemm(terms % 3 + 1)
        assert ctx.tuning()["gemm_tile"] == 64
        ctx.set_gemm(2)
        ctx.set_tiles(t["z_sticks"], 2, ctx.tuning()["gemm_tile"])
        assert np.array_equal(ctx.overlap(x, x), ref)
    ctx.close()
