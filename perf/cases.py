"""Workloads of the plane-wave SCF library, each through a public entry point.

A case is a dict with a ``kind`` and its sizes; ``prepare`` builds what a
calling program holds (the context with its plane-wave sets and potentials,
the input blocks), ``run`` makes one pass, ``work`` states the bytes and
operations a pass cannot do without, ``exact`` gives the same outputs from
numpy / torch in 64 bits where they have a closed value.

Kinds
  scf      wavefunctions initialised, then SCF steps (``steps`` of them, or
           to |dE| < 1e-6 Ha with steps = 0): what the SCF driver runs
  bands    non-self-consistent bands along a k-path at a fixed potential
  apply_h  H|psi> of host-held bands at one k-point
  density  density of host-held bands added to a host-held one
  hartree  Hartree potential and energy of a host-held density
  overlap  X^H Y on device-resident blocks
  hegv     generalised subspace problem H c = w S c, lowest eigenpairs
  heev     standard Hermitian problem, lowest eigenpairs

Outputs of a mixed-precision context are handed on in the precision of its
wavefunctions (complex64 / float32).  Eigenvectors are fixed up to a phase
only: their first component is made real and positive, as a program that
stores them would.
"""
import ctypes as C
import functools
import math
from types import SimpleNamespace

import numpy as np
import torch

from derek_amd import lib
from derek_amd.scf import Setup
from derek_amd.spectral import CUBIC_PATH, kpath

FP64, MIXED = "fp64", "mixed"


def listed():
    return [
        # overlaps of the smallest system's bands (32^3 grid, 10 bands): launch latency
        dict(name="overlap_1503x10", kind="overlap", npw=1503, m=10, n=10, herm=True),
        # a Davidson block of the largest system (2 x 300 bands against 300, 161214 plane waves)
        dict(name="overlap_161214x600x300", kind="overlap", npw=161214, m=600, n=300, herm=False),
        # the Davidson subspace problem of an 80-band and of a 300-band system
        dict(name="hegv_160", kind="hegv", n=160, nev=80),
        dict(name="hegv_600", kind="hegv", n=600, nev=300),
        # the drop-in H|psi> call of a host program, 20 bohr cell at the default grid scale (99^3)
        dict(name="apply_h_99", kind="apply_h", lx=20.0, ly=20.0, lz=20.0, ecut=30.0, gscale=2.0, nb=16,
             precision=FP64),
        # density of one k-point's bands in the mixed form, elongated cell (72 x 72 x 105 grid)
        dict(name="density_72x72x105", kind="density", lx=16.0, ly=16.0, lz=23.5, ecut=20.0, gscale=2.2, nb=24,
             precision=MIXED),
        # Hartree potential of a host program's density on the 108^3 grid
        dict(name="hartree_108", kind="hartree", lx=20.0, ly=20.0, lz=20.0, ecut=30.0, gscale=2.15, precision=FP64),
        # whole SCF of a small molecule-sized cell: many short launches
        dict(name="scf_32", kind="scf", lx=10.0, ly=10.0, lz=10.0, ecut=10.0, gscale=2.15, mp=1, nelec=8, nb=10,
             nwells=4, kT=0.005, precision=FP64, steps=0, graph=False),
        # whole SCF of the 128-electron Gamma system in FP64 (62669 plane waves, 80 bands)
        dict(name="scf_108", kind="scf", lx=20.0, ly=20.0, lz=20.0, ecut=30.0, gscale=2.15, mp=1, nelec=128, nb=80,
             nwells=16, kT=0.01, precision=FP64, steps=0, graph=False),
        # first SCF steps of a 4 x 4 x 4 mesh in the mixed form, every k-point batched, step graph
        dict(name="scf_72_mesh4_mixed", kind="scf", lx=16.0, ly=16.0, lz=16.0, ecut=20.0, gscale=2.2, mp=4, nelec=32,
             nb=24, nwells=8, kT=0.01, precision=MIXED, steps=5, graph=True),
        # band structure on a 17-point path at the default grid scale (65^3) in FP64
        dict(name="bands_65_path", kind="bands", lx=16.0, ly=16.0, lz=16.0, ecut=20.0, gscale=2.0, seg=4, nelec=32,
             nb=24, nwells=8, precision=FP64, steps=6),
        # first SCF steps of the 300-band, 8-k-point system in the mixed form (144^3)
        dict(name="scf_144_mesh2_mixed", kind="scf", lx=30.0, ly=30.0, lz=30.0, ecut=25.0, gscale=2.125, mp=2,
             nelec=512, nb=300, nwells=64, kT=0.01, precision=MIXED, steps=2, graph=False),
    ]


def _log(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def draw(rng):
    kind = rng.choice(["scf", "scf", "scf", "bands", "apply_h", "density", "hartree", "overlap", "hegv", "heev"])
    if kind == "overlap":
        m = int(round(_log(rng, 6, 600)))
        herm = rng.random() < 0.5
        n = m if herm else max(1, int(round(m * rng.choice([0.5, 1.0, rng.uniform(0.3, 1.5)]))))
        return dict(kind=kind, npw=int(_log(rng, max(700, 4 * m), 161214)), m=m, n=min(n, 600), herm=herm)
    if kind in ("hegv", "heev"):
        n = int(round(_log(rng, 12, 600)))
        return dict(kind=kind, n=n, nev=max(1, int(round(n * rng.choice([0.5, 0.5, rng.uniform(0.1, 1.0)])))))
    lx = round(_log(rng, 9.0, 24.0), 2)
    cubic = rng.random() < 0.5
    ly, lz = (lx, lx) if cubic else (round(lx * rng.uniform(0.8, 1.3), 2), round(lx * rng.uniform(0.7, 1.5), 2))
    c = dict(kind=kind, lx=lx, ly=ly, lz=lz, ecut=round(rng.uniform(10.0, 28.0), 1),
             gscale=rng.choice([2.0, 2.0, 2.1, 2.15, 2.2]), precision=rng.choice([FP64, FP64, MIXED]))
    npw = _npw(c)
    if kind in ("scf", "bands"):
        nelec = 2 * max(2, int(lx * ly * lz * rng.uniform(0.004, 0.012) / 2))
        c.update(nelec=nelec, nb=int(nelec * rng.uniform(0.58, 0.75)) + 3, nwells=max(2, nelec // 8))
        # work of one step relative to the largest system's, to bound the mesh
        most = 8 * 300 * 161214.0 * (300 + 900)
        per_k = c["nb"] * npw * (c["nb"] + 900.0) * 4
        meshes = [q for q in (1, 1, 2, 3, 4) if q ** 3 * per_k < 0.3 * most]
        if kind == "scf":
            q = rng.choice(meshes)
            c.update(mp=q, kT=rng.choice([0.005, 0.01, 0.02]), steps=rng.choice([3, 4, 6]), graph=rng.random() < 0.5)
        else:
            c.update(seg=rng.choice([2, 3, 5]), steps=rng.choice([4, 6, 8]))
    elif kind != "hartree":
        c.update(nb=int(round(_log(rng, 1, 48))))
    return c


# ---------------------------------------------------------------- discretisation
def _npw(c):
    """Plane waves of the sphere 1/2 G^2 <= ecut (its volume over that of a G cell)."""
    return c["lx"] * c["ly"] * c["lz"] * (2.0 * c["ecut"]) ** 1.5 / (6.0 * math.pi ** 2)


def _cell(c):
    return np.diag([c["lx"], c["ly"], c["lz"]])


def _dims(c):
    return lib.grid_dims(_cell(c), c["ecut"], c["gscale"])[1]


@functools.lru_cache(maxsize=16)
def _setup(lengths, ecut, gscale, mp, seg):
    """Grid, plane-wave sets and |G|^2 (the potential is set per seed)."""
    spec = SimpleNamespace(lengths=list(lengths), ecut=ecut, g_fine_scale=gscale, mp=(mp, mp, mp), centres=[],
                           heights=[], widths=[], cos_amp=0.0)
    return Setup(spec, kfrac=kpath([v for _, v in CUBIC_PATH], seg)[0] if seg else None)


def _setup_of(c):
    return _setup((c["lx"], c["ly"], c["lz"]), c["ecut"], c["gscale"], c.get("mp", 1), c.get("seg", 0))


def _context(c, su, nb):
    ctx = lib.Context(su.dims, su.nk, nb, su.volume, max(su.npw), _prec(c))
    for k in range(su.nk):
        ctx.set_basis(k, su.fft_index[k], su.kin[k], su.weights[k])
    return ctx


def _prec(c):
    return lib.DEREK_FP64 if c["precision"] == FP64 else lib.DEREK_MIXED


def _wells(c, dims, nwells, rng):
    """Periodic Gaussian wells (depth 1-3 Ha, width 0.8-1.5 bohr): a product of
    one-dimensional periodic sums per well."""
    h, w = -rng.uniform(1.0, 3.0, nwells), rng.uniform(0.8, 1.5, nwells)
    axes = []
    for n, length in zip(dims, (c["lx"], c["ly"], c["lz"])):
        d = np.arange(n)[None, :] * (length / n) - rng.uniform(0.0, length, nwells)[:, None]
        axes.append(sum(np.exp(-0.5 * ((d + s * length) / w[:, None]) ** 2) for s in (-1, 0, 1)))
    xy = (h[:, None, None] * axes[0][:, :, None] * axes[1][:, None, :]).reshape(nwells, -1)
    return np.ascontiguousarray((xy.T @ axes[2]).reshape(-1))


def _bands(kin, nb, rng):
    """Smooth random bands: plane-wave coefficients falling off with the
    kinetic energy, each band normalised."""
    p = rng.standard_normal((nb, 2 * len(kin))).view(np.complex128) / (1.0 + kin)
    return p / np.linalg.norm(p, axis=1)[:, None]


def _freq(n):
    return np.fft.fftfreq(n, 1.0 / n)


# ---------------------------------------------------------------- inputs
def prepare(case, seed):
    rng = np.random.default_rng(seed)
    c, kind = case, case["kind"]
    if kind == "overlap":
        ctx = lib.Context([8, 8, 8], 1, 1, 1.0, 1)  # the library handle and its stream
        x, y = _blocks(c, seed)
        s = torch.empty(c["n"], c["m"], dtype=torch.complex128, device="cuda")
        return dict(case=c, ctx=ctx, x=x, y=y, s=s)
    if kind in ("hegv", "heev"):
        ctx = lib.Context([8, 8, 8], 1, 1, 1.0, 1)
        s, h = _pencil(c["n"], rng)
        return dict(case=c, ctx=ctx, s=s, h=h if kind == "hegv" else 0.5 * (h + h.conj().T))
    su = _setup_of(c)
    if kind == "hartree":
        ctx = lib.Context(su.dims, 1, 1, su.volume, 1, _prec(c))
        ctx.set_gsq(su.gsq)
        return dict(case=c, ctx=ctx, rho=_rho(c, su, rng))
    if kind in ("apply_h", "density"):
        ctx = _context(c, su, c["nb"])
        psi = _bands(su.kin[0], c["nb"], rng)
        if kind == "apply_h":
            ctx.set_vloc(_wells(c, su.dims, 8, rng))
            return dict(case=c, ctx=ctx, psi=psi)
        return dict(case=c, ctx=ctx, psi=psi, occ=rng.uniform(0.0, 2.0, c["nb"]), rho=_rho(c, su, rng))
    ctx = _context(c, su, c["nb"])
    v = _wells(c, su.dims, c["nwells"], rng)
    ctx.set_gsq(su.gsq)
    ctx.set_vext(v)
    return dict(case=c, ctx=ctx, v=v, seed=seed)


def _blocks(c, seed):
    """Two blocks of nearly orthonormal vectors on the device (one and the same when herm)."""
    g = torch.Generator(device="cuda").manual_seed(seed)

    def block(m):
        return torch.randn(m, c["npw"], dtype=torch.complex128, device="cuda", generator=g) / math.sqrt(c["npw"])
    x = block(c["m"])
    return x, x if c["herm"] else block(c["n"])


def _rho(c, su, rng):
    return 0.02 - 0.05 * _wells(c, su.dims, 6, rng)


def _pencil(n, rng):
    """S = M^H M and H = M^H (D + coupling) M: the overlap and Hamiltonian of
    a nearly orthonormal block with a kinetic-like spectrum."""
    def gauss():
        return rng.standard_normal((n, 2 * n)).view(np.complex128) / math.sqrt(2.0 * n)
    m = np.eye(n) + 0.3 * gauss()
    a = gauss()
    h = np.diag(np.sort(rng.uniform(-1.0, 8.0, n))) + 0.2 * (a + a.conj().T)
    s, h = m.conj().T @ m, m.conj().T @ h @ m
    return 0.5 * (s + s.conj().T), 0.5 * (h + h.conj().T)


# ---------------------------------------------------------------- one pass
def _phase(z):
    """Columns with their first component real and positive."""
    return z * (np.conj(z[0]) / np.abs(z[0]))


def _as(c, a):
    """A mixed context's result in the precision of its wavefunctions."""
    if c["precision"] == FP64:
        return a
    t = torch.from_numpy(np.atleast_1d(np.asarray(a)))
    return t.to(torch.complex64 if t.is_complex() else torch.float32)


def run(state):
    c, ctx = state["case"], state["ctx"]
    kind = c["kind"]
    if kind == "overlap":
        lib.check(ctx.lib.derek_hip_overlap_noalloc(
            ctx.h, C.c_int64(c["npw"]), C.c_int32(c["m"]), C.c_int32(c["n"]), C.c_void_p(state["x"].data_ptr()),
            C.c_void_p(state["y"].data_ptr()), C.c_void_p(state["s"].data_ptr())))
        return state["s"]
    if kind == "hegv":
        w, z = ctx.hegv(state["s"], state["h"], c["nev"])
        return w, _phase(z)
    if kind == "heev":
        w, z = ctx.heev(state["h"], c["nev"])
        return w, _phase(z)
    if kind == "hartree":
        v, e = ctx.hartree(state["rho"])
        return _as(c, v), e
    if kind == "apply_h":
        return _as(c, ctx.apply_h(0, state["psi"]))
    if kind == "density":
        return _as(c, ctx.density(0, state["psi"], state["occ"], state["rho"]))
    if kind == "bands":
        ctx.scf_init(c["nelec"], kT=0.0, seed=state["seed"])
        ctx.set_vloc(state["v"])
        ctx.nscf(max_iter=c["steps"], res_tol=1e-9)
        return _as(c, ctx.eigenvalues())
    ctx.scf_init(c["nelec"], kT=c["kT"], seed=state["seed"], graph=c["graph"])
    e, old = [], None
    for _ in range(c["steps"] or 60):
        r = ctx.scf_step()
        e.append(r["etot"])
        if not c["steps"] and old is not None and abs(r["etot"] - old) < 1e-6 and r["refine_left"] == 0:
            break
        old = r["etot"]
    return {"etot": _as(c, np.array(e)), "eigenvalues": _as(c, ctx.eigenvalues()),
            "occupations": _as(c, ctx.occupations()), "density": _as(c, ctx.get_density())}


# ---------------------------------------------------------------- compulsory work
def _fft_flops(c, dims):
    """One inverse or forward transform of one band: z on the sphere's sticks,
    y on its x planes, x on every line; 5 n log2 n per line."""
    r = [math.sqrt(2.0 * c["ecut"]) * c[q] / (2.0 * math.pi) for q in ("lx", "ly", "lz")]
    line = [5.0 * n * math.log2(n) for n in dims]
    return (math.pi * r[0] * r[1] * line[2] + (2.0 * r[0] + 1.0) * dims[2] * line[1] + dims[1] * dims[2] * line[0])


def work(case):
    c, kind = case, case["kind"]
    if kind == "overlap":
        return {"bytes": 16.0 * c["npw"] * (c["m"] + (0 if c["herm"] else c["n"])) + 16.0 * c["m"] * c["n"],
                "flops": (4.0 if c["herm"] else 8.0) * c["npw"] * c["m"] * c["n"]}
    if kind in ("hegv", "heev"):
        # Cholesky, reduction, tridiagonalisation, back-transformation (complex operations)
        n, v = float(c["n"]), float(c["nev"])
        fl = 4.0 * (4.0 / 3.0 * n ** 3 + 2.0 * n * n * v)
        if kind == "hegv":
            fl += 4.0 * (n ** 3 / 3.0 + 2.0 * n ** 3 + n * n * v)
        return {"bytes": 16.0 * n * ((2 if kind == "hegv" else 1) * n + v) + 8.0 * v, "flops": fl}
    dims = _dims(c)
    ng, npw = float(np.prod(dims)), _npw(c)
    sc = 16.0 if c["precision"] == FP64 else 8.0
    full = 5.0 * ng * math.log2(ng)
    if kind == "hartree":
        return {"bytes": 24.0 * ng, "flops": 2.0 * full}
    nb = float(c["nb"])
    if kind == "apply_h":
        return {"bytes": 32.0 * nb * npw + 12.0 * npw + sc / 2 * ng, "flops": nb * (2.0 * _fft_flops(c, dims) + 2.0 * ng)}
    if kind == "density":
        return {"bytes": 16.0 * nb * npw + 12.0 * npw + 16.0 * ng, "flops": nb * (_fft_flops(c, dims) + 4.0 * ng)}
    nk = float(c["mp"] ** 3 if kind == "scf" else 4 * c["seg"] + 1)
    hpsi_b, hpsi_f = 2.0 * npw * sc + 12.0 * npw + ng * sc / 2 / nb, 2.0 * _fft_flops(c, dims) + 2.0 * ng
    if kind == "bands":
        its, steps, dens = 1.0 + c["steps"], 1.0, 0.0
        gemm = nk * 8.0 * npw * nb * nb * (3.0 + 12.0 * c["steps"])
    else:
        steps = float(c["steps"] or 15)
        its, dens = 3.0 * steps + 2.0, steps  # H X and two Davidson steps each, four in the first step
        gemm = nk * 8.0 * npw * nb * nb * (3.0 * steps + 12.0 * (2.0 * steps + 2.0))
    grid = 384.0 * ng * dens
    return {"bytes": nk * nb * (its * hpsi_b + dens * npw * sc) + grid,
            "flops": gemm + nk * nb * (its * hpsi_f + dens * (_fft_flops(c, dims) + 4.0 * ng)) + 6.0 * dens * full}


# ---------------------------------------------------------------- 64-bit values
def _on_grid(psi, index, dims):
    """Bands on the real-space grid, sum_G c(G) e^{iGr} (z fastest)."""
    g = torch.zeros(psi.shape[0], int(np.prod(dims)), dtype=torch.complex128)
    g[:, torch.from_numpy(index.astype(np.int64))] = torch.from_numpy(psi)
    return torch.fft.ifftn(g.reshape(-1, *dims), dim=(1, 2, 3), norm="forward")


def _waves(c, dims):
    """Plane waves 1/2 G^2 <= ecut in the order x outer, z inner, m from -n/2 up: FFT bin, kinetic energy."""
    m = [np.arange(-(n // 2), n - n // 2) for n in dims]
    g = [2.0 * math.pi * q / length for q, length in zip(m, (c["lx"], c["ly"], c["lz"]))]
    t = 0.5 * (g[0][:, None, None] ** 2 + g[1][None, :, None] ** 2 + g[2][None, None, :] ** 2)
    i = np.nonzero(t <= c["ecut"])
    b = [m[a][i[a]] % dims[a] for a in range(3)]
    return (b[0] * dims[1] + b[1]) * dims[2] + b[2], t[i]


def exact(case, seed):
    c, kind = case, case["kind"]
    if kind in ("scf", "bands"):
        return None
    rng = np.random.default_rng(seed)
    if kind == "overlap":
        x, y = _blocks(c, seed)
        return (x.conj() @ y.transpose(0, 1).contiguous()).transpose(0, 1).contiguous()
    if kind in ("hegv", "heev"):
        s, h = _pencil(c["n"], rng)
        if kind == "heev":
            w, z = np.linalg.eigh(0.5 * (h + h.conj().T))
        else:
            li = np.linalg.inv(np.linalg.cholesky(s))
            a = li @ h @ li.conj().T
            w, z = np.linalg.eigh(0.5 * (a + a.conj().T))
            z = li.conj().T @ z
        return w[:c["nev"]], _phase(z[:, :c["nev"]])
    dims = _dims(c)
    volume = c["lx"] * c["ly"] * c["lz"]
    if kind == "hartree":
        rho = torch.from_numpy(_rho(c, SimpleNamespace(dims=dims), rng)).reshape(*dims)
        g = [(2.0 * math.pi / length * torch.from_numpy(_freq(n))) ** 2
             for n, length in zip(dims, (c["lx"], c["ly"], c["lz"]))]
        gsq = g[0][:, None, None] + g[1][None, :, None] + g[2][None, None, :]
        k = 4.0 * math.pi / torch.where(gsq > 0, gsq, torch.inf)
        v = torch.fft.ifftn(torch.fft.fftn(rho.to(torch.complex128)) * k).real.contiguous()
        return v.reshape(-1), float(0.5 * volume / v.numel() * (v * rho).sum())
    index, kin = _waves(c, dims)
    psi = _bands(kin, c["nb"], rng)
    if kind == "apply_h":
        v = torch.from_numpy(_wells(c, dims, 8, rng)).reshape(*dims)
        out = np.empty_like(psi)
        for b in range(0, c["nb"], 4):
            h = torch.fft.fftn(v * _on_grid(psi[b:b + 4], index, dims), dim=(1, 2, 3), norm="forward")
            out[b:b + 4] = kin * psi[b:b + 4] + h.reshape(h.shape[0], -1)[:, torch.from_numpy(index)].numpy()
        return out
    occ = rng.uniform(0.0, 2.0, c["nb"])
    rho = torch.from_numpy(_rho(c, SimpleNamespace(dims=dims), rng)).reshape(*dims)
    for b in range(c["nb"]):
        rho = rho + occ[b] / volume * _on_grid(psi[b:b + 1], index, dims)[0].abs() ** 2
    return rho.reshape(-1)
