"""The mixing system for every shape of its elimination (a row per lane, four
lanes per row; 1 to 16 slots): the SCF with other history lengths than the
default of 8 against the oracle's with the same length.

Bounds: those of the other SCF comparisons, 1e-7 Ha and 1e-6 of the largest
density, at |dE| < 1e-11 and ||rho_out - rho_in|| < 1e-8 on both sides.
"""
import numpy as np
import pytest

from derek_amd import config
from derek_amd import scf as gscf
from oracle import scf as oscf
from tests.conftest import oracle_system

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("history", [2, 3, 5, 16])
def test_history_lengths_match_oracle(history):
    print("pulay history", history, flush=True)
    spec = config.small_system(seed=13, mp=(2, 1, 1), kT=0.01, nelec=6, nbands=8)
    setup = gscf.Setup(spec)
    ctx = setup.context()
    res = gscf.run(spec, max_scf=60, energy_tol=1e-11, rho_tol=1e-8, history=history, setup=setup, ctx=ctx, log=print)
    rho = ctx.get_density()
    ctx.close()
    ref = oscf.scf(oracle_system(spec), max_scf=60, energy_tol=1e-11, rho_tol=1e-8, history=history)
    assert res["converged"] and ref["converged"]
    assert abs(res["etot"] - ref["etot"]) < 1e-7
    assert np.max(np.abs(rho - ref["rho_out"])) < 1e-6 * np.max(ref["rho_out"])
