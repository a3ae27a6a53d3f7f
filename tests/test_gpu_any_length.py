"""H|psi> and the density at FFT lengths without kernels of their own, against
the oracle: every radix from 1 to 16 in both stages of a length r1 * r2, axes
of different lengths, column tiles and stick blocks with remainders, active
rows in any order, and the lengths that have no such split (Stockham).

An FFT of n points carries a relative rounding error of a few eps * log2(n)
(eps = 1.1e-16 / 6e-8), at most 30 eps here for inverse, multiply and forward
together; the bounds are the ones of the other pipeline tests, 1e-12 and 5e-5
of the largest value.
"""
import numpy as np
import pytest

from derek_amd import lib
from oracle import ks as oks
from tests.conftest import assert_close

pytestmark = pytest.mark.gpu

DIMS = [(1, 2, 3), (5, 7, 4), (8, 6, 13), (22, 26, 10), (65, 33, 30), (16, 15, 210), (28, 98, 11), (99, 40, 24),
        (50, 63, 64), (140, 21, 39), (12, 225, 18), (45, 14, 240), (256, 9, 91), (65, 65, 65), (54, 54, 36),
        (125, 8, 162), (35, 147, 20)]


def waves(dims, rng, share=0.3):
    """A random set of FFT bins on a few columns, in shuffled order."""
    nx, ny, nz = dims
    xs = rng.permutation(nx)[:max(1, int(share * 1.5 * nx))]
    idx = []
    for x in xs:
        for y in rng.permutation(ny)[:max(1, int(share * ny))]:
            z = rng.permutation(nz)[:max(1, int(share * nz))]
            idx.append((x * ny + y) * nz + z)
    return rng.permutation(np.concatenate(idx)).astype(np.int32)


@pytest.mark.parametrize("dims", DIMS)
@pytest.mark.parametrize("precision", [lib.DEREK_FP64, lib.DEREK_MIXED])
def test_any_length_apply_h_and_density(dims, precision):
    rng = np.random.default_rng(sum(dims))
    nb, volume, weight = 5, 37.0, 0.7
    sets = [waves(dims, rng), waves(dims, rng, 0.2)]
    kins = [rng.uniform(0.0, 3.0, len(s)) for s in sets]
    v = rng.normal(size=int(np.prod(dims)))
    tol = 1e-12 if precision == lib.DEREK_FP64 else 5e-5
    ctx = lib.Context(list(dims), 2, nb, volume, max(len(s) for s in sets), precision)
    for k in range(2):
        ctx.set_basis(k, sets[k], kins[k], weight)
    ctx.set_vloc(v)
    for zs in (16, 32):
        print("any length", dims, precision, "sticks", zs, flush=True)
        ctx.set_tiles(zs, 2, 64)
        ctx.set_launch(bands_per_wg=2, items_per_launch=3, fused=zs == 16)
        for k in range(2):
            psi = rng.normal(size=(nb, len(sets[k]))) + 1j * rng.normal(size=(nb, len(sets[k])))
            assert_close(ctx.apply_h(k, psi), oks.apply_h(psi, sets[k], kins[k], v, dims), tol, f"H psi k={k}")
            occ = np.array([2.0, 0.0, 1.3, 0.4, 2.0])
            r0 = rng.uniform(size=v.size)
            ref = r0 + oks.density([psi], [occ], [weight], [sets[k]], dims, volume)
            assert_close(ctx.density(k, psi, occ, r0), ref, tol, f"density k={k}")
    ctx.close()


def outer(n, rng):
    """Bins of the outer quarters (b < n/4, b >= 3n/4), the edges always among them."""
    b = np.array([q for q in range(n) if 4 * q < n or 4 * q >= 3 * n])
    return np.union1d(b[[0, -1, (n + 3) // 4 - 1]], rng.permutation(b)[:max(1, len(b) // 2)])


@pytest.mark.parametrize("dims", DIMS[:-1] + [(72, 72, 105), (32, 32, 65), (108, 108, 21), (144, 144, 10)])
@pytest.mark.parametrize("precision", [lib.DEREK_FP64, lib.DEREK_MIXED])
@pytest.mark.parametrize("quarter", [True, False])
def test_outer_quarters(dims, precision, quarter):
    """Plane waves in the outer quarters of every axis take the transforms with
    dropped zero inputs and unread outputs, separate and fused; a single bin
    outside them (quarter False) takes the full ones."""
    rng = np.random.default_rng(sum(dims) + 1)
    nx, ny, nz = dims
    idx = np.concatenate([(x * ny + y) * nz + outer(nz, rng) for x in outer(nx, rng) for y in outer(ny, rng)])
    if not quarter:
        idx = np.append(idx, ((nx // 2) * ny + ny // 2) * nz + nz // 2)
    idx = rng.permutation(np.unique(idx)).astype(np.int32)[:6000]
    nb, volume, weight = 3, 21.0, 0.9
    kin = rng.uniform(0.0, 3.0, len(idx))
    v = rng.normal(size=nx * ny * nz)
    tol = 1e-12 if precision == lib.DEREK_FP64 else 5e-5
    ctx = lib.Context(list(dims), 1, nb, volume, len(idx), precision)
    ctx.set_basis(0, idx, kin, weight)
    ctx.set_vloc(v)
    psi = rng.normal(size=(nb, len(idx))) + 1j * rng.normal(size=(nb, len(idx)))
    occ = np.array([2.0, 1.3, 0.4])
    ref = oks.apply_h(psi, idx, kin, v, dims)
    rref = oks.density([psi], [occ], [weight], [idx], dims, volume)
    for fused in (True, False):
        print("outer quarters", dims, precision, quarter, "fused", fused, flush=True)
        ctx.set_launch(bands_per_wg=2, items_per_launch=256, fused=fused)
        assert_close(ctx.apply_h(0, psi), ref, tol, "H psi")
        assert_close(ctx.density(0, psi, occ), rref, tol, "density")
    ctx.close()


@pytest.mark.parametrize("n", [72, 108, 144])
@pytest.mark.parametrize("planes", [27, 28, 29, 45, 56, 57, 70, 76, 108])
@pytest.mark.parametrize("precision", [lib.DEREK_FP64, lib.DEREK_MIXED])
def test_fused_pass_plane_counts(n, planes, precision):
    """Active x planes at the edges of the fused pass: groups of planes per
    wavefront, wavefronts that the LDS holds, and the switches to the barrier
    kernel and to the separate passes."""
    planes, nz = min(planes, n), 6
    rng = np.random.default_rng(n + planes)
    xs = rng.permutation(n)[:planes]
    idx = np.concatenate([(x * n + y) * nz + np.arange(0, nz, 1 + y % 3) for x in xs for y in rng.permutation(n)[:3]])
    idx = rng.permutation(np.unique(idx)).astype(np.int32)
    kin = rng.uniform(0.0, 3.0, len(idx))
    v = rng.normal(size=n * n * nz)
    tol = 1e-12 if precision == lib.DEREK_FP64 else 5e-5
    print("planes", n, planes, precision, flush=True)
    ctx = lib.Context([n, n, nz], 1, 2, 13.0, len(idx), precision)
    ctx.set_basis(0, idx, kin, 1.1)
    ctx.set_vloc(v)
    psi = rng.normal(size=(2, len(idx))) + 1j * rng.normal(size=(2, len(idx)))
    occ = np.array([2.0, 0.7])
    assert_close(ctx.apply_h(0, psi), oks.apply_h(psi, idx, kin, v, (n, n, nz)), tol, "H psi")
    assert_close(ctx.density(0, psi, occ), oks.density([psi], [occ], [1.1], [idx], (n, n, nz), 13.0), tol, "density")
    ctx.close()
