"""Performance cases: the runs a treatment-planning program has this framework do.

Each case goes through the Python entry points over the C ABI (``Context``,
``Context.run_dosxyz``, ``Context.run_dosxyz_noalloc``, ``Context.run_dij``,
``Context.dij_assemble``, ``Server``) as a program would call them, with the
physics tables and the phantom already resident.  A case is a dict of plain
values; ``listed()`` gives the fixed ones, ``draw(rng)`` one more of the same
ranges, ``prepare`` the inputs of a seed, ``run`` one pass, ``work`` the bytes
and operations a pass cannot do without, and ``exact`` the result in plain
64-bit numpy where one exists.

Transport cases have no such result (a Monte Carlo estimate depends on every
particle's random stream), so ``exact`` gives one for the matrix assembly only.
"""
import functools
import math

import numpy as np
import torch

import ompmc_amd as omc
from ompmc_amd import phantoms as P

NBATCH = 10              # statistical batches of every run, as in the sample inputs

# Operations of one history, to the order of magnitude: a 6 MV photon's few
# interactions and the ~30 condensed-history steps of its electrons at about
# two thousand each, and a step per ~60 keV of a primary electron.
PHOTON_FLOPS = 6.0e4
STEP_FLOPS = 2.0e3

# Matrix entries above 1e-4 of the beamlet's maximum, per history (measured on
# the 1960-beamlet plan; fewer histories per beamlet leave more of them).
ENTRIES_PER_HISTORY = 1.9


def listed():
    return [
        # a first look: the smallest dose run somebody waits for, all latency
        dict(name="dose_water32_1e4", kind="dose", phantom="water", nx=32, ny=32, nz=32, voxel=0.5, energy=2.0,
             histories=10_000, precision=32, charge=0, nsplit=1, field=5.0),
        # the reference's plain case: 2 MeV parallel beam on 60^3 water, FP64 throughout
        dict(name="dose_water60_1e6_fp64", kind="dose", phantom="water", nx=60, ny=60, nz=60, voxel=0.5, energy=2.0,
             histories=1_000_000, precision=64, charge=0, nsplit=1, field=10.0),
        # the heterogeneous slab with a 6 MV spectrum at its full 1e7 histories
        dict(name="dose_slab128_1e7", kind="dose", phantom="slab", nx=128, ny=128, nz=128, voxel=0.3, energy=0.0,
             histories=10_000_000, precision=32, charge=0, nsplit=1, field=10.0),
        # an electron field on a CT: every primary is a charged particle
        dict(name="dose_ct_electrons_2e5", kind="dose", phantom="ct", nx=96, ny=96, nz=64, voxel=0.3, energy=9.0,
             histories=200_000, precision=32, charge=-1, nsplit=1, field=6.0),
        # photon splitting at the sample input's factor, on a grid of odd sizes
        dict(name="dose_ct_odd_split20_1e5", kind="dose", phantom="ct", nx=101, ny=97, nz=83, voxel=0.27, energy=0.0,
             histories=100_000, precision=32, charge=0, nsplit=20, field=7.0),
        # the history form into device buffers, for callers that cannot allocate
        dict(name="dose_noalloc_1e5", kind="noalloc", phantom="slab", nx=64, ny=64, nz=64, voxel=0.45, energy=0.0,
             histories=100_000, precision=32, charge=0, nsplit=1, field=8.0),
        # one beam's matrix on a small CT while a plan is being set up
        dict(name="dij_one_beam_2e4", kind="dij", nx=64, ny=64, nz=48, voxel=0.4, nbeams=1, radius=1.3, every=1,
             per_beamlet=1000, precision=32, gaussian=False, var=False, room=8.0),
        # the five-beam plan: 1960 beamlets of lognormal histories, the whole matrix in host memory
        dict(name="dij_plan_1960", kind="dij", nx=160, ny=160, nz=100, voxel=0.25, nbeams=5, radius=5.6, every=1,
             per_beamlet=7000, precision=32, gaussian=False, var=False, room=3.0),
        # a tenth of that plan in FP64 with a Gaussian spot and the variance matrix
        dict(name="dij_plan_196_fp64_var", kind="dij", nx=160, ny=160, nz=100, voxel=0.25, nbeams=5, radius=5.6,
             every=10, per_beamlet=7000, precision=64, gaussian=True, var=True, room=8.0),
        # every 200th beamlet of a nine-beam plan on a fine grid: 13 M voxels, few beamlets, many histories each
        dict(name="dij_large_grid_50", kind="dij", nx=256, ny=256, nz=200, voxel=0.2, nbeams=9, radius=9.4,
             every=200, per_beamlet=12000, precision=32, gaussian=False, var=False, room=8.0),
        # the matrix from tallies made elsewhere
        dict(name="assemble_12x10", kind="assemble", nx=48, ny=48, nz=40, voxel=0.5, nbeamlets=12),
        # a resident server with small and middling dose and matrix requests in flight together
        dict(name="serve_8_requests", kind="serve", nx=72, ny=72, nz=64, voxel=0.35, requests=8, smallest=100_000,
             largest=1_500_000),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(("dose", "dose", "dose", "dij", "dij", "noalloc", "assemble", "serve"))
    if kind in ("dose", "noalloc"):
        phantom = rng.choice(("water", "slab", "ct"))
        nx, nz = rng.randint(30, 128), rng.randint(30, 128)
        precision = rng.choice((32, 32, 32, 64))
        charge = rng.choice((0, 0, 0, -1, 1)) if kind == "dose" else 0
        nsplit = rng.choice((1, 1, 1, 4, 20)) if kind == "dose" and charge == 0 else 1
        energy = round(rng.uniform(4.0, 12.0), 2) if charge else rng.choice((0.0, 0.0, round(rng.uniform(0.5, 10.0), 2)))
        most = 4_000_000 if kind == "dose" else 200_000
        most //= (2 if precision == 64 else 1) * (1 if charge == 0 else 8) * nsplit
        return dict(kind=kind, phantom=phantom, nx=nx, ny=nx if phantom != "ct" else rng.randint(30, 128),
                    nz=nx if phantom != "ct" else nz, voxel=round(rng.uniform(0.2, 0.5), 3), energy=energy,
                    histories=max(10 * NBATCH, _log_int(rng, 8_000, most)), precision=precision, charge=charge,
                    nsplit=nsplit, field=round(rng.uniform(2.0, 6.0), 2))
    if kind == "dij":
        return dict(kind=kind, nx=rng.randint(48, 160), ny=rng.randint(48, 160), nz=rng.randint(40, 120),
                    voxel=round(rng.uniform(0.2, 0.4), 3), nbeams=rng.randint(1, 9),
                    radius=round(rng.uniform(0.8, 2.5), 2), every=rng.choice((1, 1, 2, 3)),
                    per_beamlet=_log_int(rng, 500, 10_000), precision=rng.choice((32, 32, 64)),
                    gaussian=rng.random() < 0.3, var=rng.random() < 0.3, room=8.0)
    if kind == "assemble":
        return dict(kind=kind, nx=rng.randint(20, 60), ny=rng.randint(20, 60), nz=rng.randint(20, 48),
                    voxel=round(rng.uniform(0.25, 0.5), 3), nbeamlets=rng.randint(1, 14))
    return dict(kind=kind, nx=rng.randint(64, 128), ny=rng.randint(64, 128), nz=rng.randint(48, 96),
                voxel=round(rng.uniform(0.2, 0.5), 3), requests=rng.randint(2, 8), smallest=50_000,
                largest=_log_int(rng, 200_000, 1_500_000))


# ------------------------------------------------------------------ inputs
@functools.lru_cache(maxsize=None)
def _context(media):
    """The resident physics tables a program keeps for its media."""
    return omc.Context(list(media), device=0)


@functools.lru_cache(maxsize=4)
def _base(kind, nx, ny, nz, voxel):
    if kind == "ct":
        return P.synthetic_ct(nx=nx, ny=ny, nz=nz, vx=voxel, vy=voxel, vz=voxel, target_radius=min(2.0, 0.2 * nx * voxel))
    return P.water_cube(nx, voxel) if kind == "water" else P.slab_phantom(nx, voxel)


def _phantom(kind, case, seed):
    """The phantom of a seed: on a CT and in the slabs every voxel's density
    varies by up to 1%, as reconstructed densities do."""
    b = _base(kind, case["nx"], case["ny"], case["nz"], case["voxel"])
    rho = b.rho
    if kind != "water":
        noise = np.random.default_rng(seed).random(rho.size, dtype=np.float32).reshape(rho.shape)
        rho = rho * (0.99 + 0.02 * noise)
    return P.Phantom(b.media, b.xb, b.yb, b.zb, b.med, rho, b.name)


def _spectrum(case, seed):
    if case.get("energy", 0.0) > 0.0:
        return omc.Spectrum.mono(case["energy"])
    return omc.Spectrum.from_histogram(*P.synthetic_6mv(seed=seed))


@functools.lru_cache(maxsize=8)
def _geometry(nbeams, radius, every):
    b = P.beamlets(nbeams=nbeams, radius=radius)
    keep = slice(every // 2, None, every) if b.n > every else slice(None)
    return b.ibeam[keep], b.src, b.corner[keep], b.side1[keep], b.side2[keep]


def _beamlets(nbeams, radius, every, per_beamlet, seed):
    """A plan's beamlets with lognormal histories around `per_beamlet`."""
    ib, src, cor, s1, s2 = _geometry(nbeams, radius, every)
    lg = np.random.default_rng(seed).normal(math.log10(per_beamlet), 0.35, len(ib))
    nh = np.clip(np.rint(10.0 ** lg), per_beamlet / 7.0, per_beamlet * 7.0).astype(np.int64)
    return P.Beamlets(ib, src, cor, s1, s2, np.maximum(nh, NBATCH))


class _Matrix:
    """The program's own arrays for a matrix: the number of entries depends on
    the histories, so it keeps room for the most it expects, zeros at the end."""

    def __init__(self, ncols, most):
        self.jc, self.ir, self.val = np.zeros(ncols + 1, np.int64), np.zeros(most, np.int64), np.zeros(most)
        self.nnz = 0

    def take(self, csc):
        jc, ir, val = csc
        n = len(ir)
        self.jc[:], self.ir[:n], self.val[:n] = jc, ir, val
        if n < self.nnz:
            self.ir[n:self.nnz], self.val[n:self.nnz] = 0, 0.0
        self.nnz = n
        return {"jc": self.jc, "ir": self.ir, "val": self.val}


class _State:
    """What the program holds before the call; releases it when dropped."""

    def __init__(self, case, seed):
        self.case, self.seed, self.phantom, self.server = case, seed, None, None

    def __del__(self):
        try:
            if self.server is not None:
                self.server.close()
            if self.phantom is not None:
                self.phantom.release()
        except Exception:
            pass


def prepare(case, seed):
    s = _State(case, seed)
    kind = case["kind"]
    ph = _phantom(case.get("phantom", "ct"), case, seed)
    s.ctx = _context(tuple(ph.media))
    s.spectrum = _spectrum(case, seed)
    if kind == "serve":
        _prepare_serve(s, ph)
        return s
    s.phantom = s.ctx.phantom(ph)
    if kind == "dij":
        s.beamlets = _beamlets(case["nbeams"], case["radius"], case["every"], case["per_beamlet"], seed)
        n = s.beamlets.n
        most = n * min(ph.nvox, int(case["room"] * 1.4 * case["per_beamlet"]))
        s.dij, s.var = _Matrix(n, most), _Matrix(n, most) if case["var"] else None
    elif kind == "assemble":
        s.endep, s.nper = _tallies(case, seed), np.full(case["nbeamlets"], 700, np.int64)
        s.dij, s.var = (_Matrix(case["nbeamlets"], case["nbeamlets"] * ph.nvox) for _ in range(2))
    elif kind == "noalloc":
        s.sum = torch.zeros(s.phantom.nreg, dtype=torch.float64, device="cuda:0")
        s.sum2 = torch.zeros_like(s.sum)
    return s


def _prepare_serve(s, ph):
    case, rng = s.case, np.random.default_rng(s.seed)
    s.server = omc.Server(s.ctx, max_inflight=4)
    half = 0.2 * case["nx"] * case["voxel"]
    s.requests, s.matrices = [], {}
    for i in range(case["requests"]):
        # the request sizes are the case's (log-spaced, small and large mixed), their streams the seed's
        f = ((i * 5) % case["requests"]) / max(1, case["requests"] - 1)
        nh = int(case["smallest"] * (case["largest"] / case["smallest"]) ** f)
        kw = dict(nbatch=NBATCH, seed=int(rng.integers(1 << 40)))
        if i % 2 == 0:
            s.requests.append(("dose", ph, dict(kw, nperbatch=nh // NBATCH, collimator=(-half, half, -half, half))))
        else:
            bix = _beamlets(1 + i % 5, 1.3, 1, 1000, s.seed + i)
            bix.nhist = np.full(bix.n, max(NBATCH, nh // bix.n), np.int64)
            s.requests.append(("dij", ph, dict(kw, bix=bix)))
            s.matrices[i] = _Matrix(bix.n, bix.n * min(ph.nvox, 8 * int(bix.nhist[0])))


def _tallies(case, seed):
    """Batch tallies of beamlets through the grid: energy falls off along z and
    across the ray, most voxels receive none, and batches scatter around the mean."""
    rng = np.random.default_rng(seed)
    nx, ny, nz, nb = case["nx"], case["ny"], case["nz"], case["nbeamlets"]
    x, y = np.arange(nx) - 0.5 * (nx - 1), np.arange(ny) - 0.5 * (ny - 1)
    z = np.exp(-0.03 * np.arange(nz))
    e = np.zeros((nb, NBATCH, nx * ny * nz + 1))
    for b in range(nb):
        cx, cy = rng.uniform(-0.3, 0.3) * nx, rng.uniform(-0.3, 0.3) * ny
        r2 = (x[None, :] - cx) ** 2 + (y[:, None] - cy) ** 2
        near = np.flatnonzero(r2.reshape(-1) < (0.2 * min(nx, ny)) ** 2)
        lat = np.exp(-0.5 * np.sqrt(r2.reshape(-1)[near]))
        mean = (z[:, None] * lat[None, :]).reshape(-1)
        at = (1 + near[None, :] + nx * ny * np.arange(nz)[:, None]).reshape(-1)
        e[b][:, at] = mean * rng.exponential(1.0, (NBATCH, mean.size))
    return e


# ------------------------------------------------------------------ one pass
def run(s):
    case, kind = s.case, s.case["kind"]
    if kind in ("dose", "noalloc"):
        h = 0.5 * case["field"]
        kw = dict(collimator=(-h, h, -h, h), charge=case["charge"], nsplit=case["nsplit"], seed=s.seed + 1,
                  precision=case["precision"])
        nper = case["histories"] // NBATCH
        if kind == "noalloc":
            s.ctx.run_dosxyz_noalloc(s.phantom, s.spectrum, nper, NBATCH, s.sum.data_ptr(), s.sum2.data_ptr(), **kw)
            return {"sum": s.sum, "sum2": s.sum2}
        e, e2, _ = s.ctx.run_dosxyz(s.phantom, s.spectrum, nper, NBATCH, **kw)
        return {"sum": e, "sum2": e2}
    if kind == "dij":
        dij, var, _, _ = s.ctx.run_dij(s.phantom, s.spectrum, s.beamlets, nbatch=NBATCH, want_var=case["var"],
                                       gaussian=case["gaussian"], sigma=0.2 if case["gaussian"] else 0.0,
                                       precision=case["precision"], seed=s.seed + 1)
        return {"dij": s.dij.take(dij), "var": s.var.take(var) if s.var else None}
    if kind == "assemble":
        dij, var, _ = s.ctx.dij_assemble(s.phantom, s.endep, s.nper)
        return {"dij": s.dij.take(dij), "var": s.var.take(var)}
    ids = []
    for what, ph, kw in s.requests:
        submit = s.server.submit_dose if what == "dose" else s.server.submit_dij
        ids.append(submit(ph, s.spectrum, **kw))
    out = []
    for k, ((what, _, _), i) in enumerate(zip(s.requests, ids)):
        r = s.server.wait(i)
        if r["error"]:
            raise RuntimeError(r["message"])
        out.append({"sum": r["sum"], "sum2": r["sum2"]} if what == "dose" else s.matrices[k].take(r["dij"]))
    return out


# ------------------------------------------------------------------ what a pass cannot do without
def work(case):
    """Bytes: the phantom (one byte of medium and four of density a voxel) read
    once, and the outputs (two FP64 sums a region, or a row index and a value a
    matrix entry) written once.  Operations: the histories'."""
    nvox = case["nx"] * case["ny"] * case["nz"]
    phantom, kind = 5.0 * nvox, case["kind"]
    if kind in ("dose", "noalloc"):
        per = STEP_FLOPS * case["energy"] / 0.06 if case["charge"] else PHOTON_FLOPS * (1 + 0.5 * (case["nsplit"] - 1))
        return {"bytes": phantom + 16.0 * nvox, "flops": case["histories"] * per}
    if kind == "dij":
        n = len(_geometry(case["nbeams"], case["radius"], case["every"])[0])
        histories = n * case["per_beamlet"] * 1.38          # the mean of the lognormal
        entries = ENTRIES_PER_HISTORY * histories * (2 if case["var"] else 1)
        return {"bytes": phantom + 16.0 * entries, "flops": histories * PHOTON_FLOPS}
    if kind == "assemble":
        n = case["nbeamlets"] * NBATCH * nvox
        return {"bytes": 8.0 * n, "flops": 4.0 * n}
    q = case["requests"]
    lo, hi = case["smallest"], case["largest"]
    mean = (hi - lo) / math.log(hi / lo) if hi > lo else lo
    return {"bytes": q * (phantom + 16.0 * nvox), "flops": q * mean * PHOTON_FLOPS}


# ------------------------------------------------------------------ the result in 64 bits
def exact(case, seed):
    """The assembly in plain numpy: per beamlet the batch means and the sum of
    their squares, the dose per history and its variance with the previous
    beamlet's variance carried in, and the entries strictly above 1e-4 of the
    maximum.  A transported dose has no value but its own random streams'."""
    if case["kind"] != "assemble":
        return None
    ph = _phantom("ct", case, seed)
    rho = ph.rho.reshape(-1)
    dx, dy, dz = (np.diff(b) for b in (ph.xb, ph.yb, ph.zb))
    vol = (dz[:, None, None] * dy[None, :, None] * dx[None, None, :]).reshape(-1)
    factor = 1.602e-10 / (vol * rho)
    e, nper, nb = _tallies(case, seed)[:, :, 1:], 700.0, float(NBATCH)
    carry, n = np.zeros(rho.size), 0
    val, var = np.zeros(e.shape[0] * rho.size), np.zeros(e.shape[0] * rho.size)
    for b in range(e.shape[0]):
        x = e[b] / nper
        dose = x.sum(0) * factor / nb
        u = ((carry + (x * x).sum(0)) * factor * factor / (nb - 1.0) - dose * dose) / nb
        off = (dose == 0.0) | (rho < 0.044)
        dose[off], u[off] = 0.0, 0.0
        carry = u
        sel = dose > 1e-4 * dose.max()
        m = n + int(sel.sum())
        val[n:m], var[n:m], n = dose[sel], u[sel], m
    return {"dij": {"jc": None, "ir": None, "val": val}, "var": {"jc": None, "ir": None, "val": var}}
