"""The work a user of this framework has it do, as timed cases.

Families (a case's "family"):
  driver   a molecular-dynamics run of the ExaMiniMD driver (examinimd_amd.App):
           the atoms come from a restart file, one pass advances the run by
           `steps` steps (thermo output and list rebuilds as the deck says) and
           takes the positions, velocities and forces.
  modules  the same time step called module by module through the C ABI, as a
           host program with its own driver does, with the atoms handed over
           and taken back in device memory.
  eval     forces and energies of a configuration the program has not seen
           before (labelling or validating a SNAP potential): positions in,
           neighbour list, forces, per-atom energies out.
  batch    an ensemble of uneven periodic replicas advanced together
           (examinimd_amd.batch.Batch), sampled after `steps` steps.
  fit_snap, fit_lj
           loss and gradient of a force-matching fit over a set of
           configurations, at one parameter set (examinimd_amd.forcematch).

listed() names what each case stands for.  Positions are lattices with
Gaussian thermal displacements and velocities are Maxwell-Boltzmann, both
from the seed; the lattices, densities, temperatures, cutoffs, skins, time
steps and rebuild intervals are those of the repository's decks and benchmark.
exact() is the same physics in torch, 64 bits, without this repository's code.
"""
import ctypes as C
import math
import os
import struct
import tempfile

import numpy as np
import torch

import examinimd_amd as emd
from examinimd_amd import batch, decks, flopcount, forcematch
from examinimd_amd.abi import (EMD_FP64, EMD_LAYOUT_RIGHT, EMD_MIXED, EMD_NEIGH_2D, EMD_NEIGH_CSR,
                               EmdBins, EmdHalo, EmdLJParams, EmdNeigh, EmdSnapParams, EmdSystem,
                               EmdVec3View)

LJ_RC, LJ_SKIN, LJ_DT, LJ_T = 2.5, 0.3, 0.005, 1.44
LJ_RHO = 0.8442
LJ_A = (4.0 / LJ_RHO) ** (1.0 / 3.0)
W_A, W_MASS, W_T, W_DT, W_SKIN = 3.1803, 183.84, 300.0, 0.0005, 1.0
W_RC, W_RFAC0 = 4.73442, 0.99363
METAL_KB, METAL_MVV2E = 8.617343e-5, 1.0364269e-4


def listed():
    return [
        # A small melt with the reference deck's output every ten steps: tutorials, tests and
        # parameter scans; launches, waits and thermo sums count.
        {"name": "melt_864", "family": "driver", "pair": "lj", "nx": 6, "ny": 6, "nz": 6,
         "precision": "fp64", "neigh": "2D", "half": False, "thermo": 10, "every": 20,
         "steps": 100},
        # The plain 32 000-atom melt of the parity runs, compressed rows, no output.
        {"name": "melt_32k_csr", "family": "driver", "pair": "lj", "nx": 20, "ny": 20, "nz": 20,
         "precision": "fp64", "neigh": "CSR", "half": False, "thermo": 0, "every": 20,
         "steps": 100},
        # The size and output rate of the reference's LJ deck, in mixed precision.
        {"name": "melt_256k_mixed", "family": "driver", "pair": "lj", "nx": 40, "ny": 40,
         "nz": 40, "precision": "mixed", "neigh": "2D", "half": False, "thermo": 10, "every": 20,
         "steps": 40},
        # Half lists with Newton's third law (--force-iteration NEIGH_HALF, newton on), an
        # uneven box.
        {"name": "melt_half_86k", "family": "driver", "pair": "lj", "nx": 25, "ny": 29, "nz": 30,
         "precision": "fp64", "neigh": "CSR", "half": True, "thermo": 0, "every": 20,
         "steps": 20},
        # The headline melt: four million atoms, mixed precision, one rebuild period.
        {"name": "melt_4m_mixed", "family": "modules", "nx": 100, "ny": 100, "nz": 100,
         "precision": "mixed", "neigh": "2D", "every": 20, "steps": 20},
        # SNAP tungsten as the reference's SNAP decks run it: a few hundred atoms, the list
        # rebuilt on every step, output every ten.
        {"name": "snap_420_every1", "family": "driver", "pair": "snap", "nx": 5, "ny": 6, "nz": 7,
         "precision": "fp64", "neigh": "CSR", "half": False, "thermo": 10, "every": 1,
         "steps": 20, "twojmax": 8},
        # The headline SNAP run: 2 000 atoms, mixed precision.
        {"name": "snap_2k_mixed", "family": "driver", "pair": "snap", "nx": 10, "ny": 10,
         "nz": 10, "precision": "mixed", "neigh": "CSR", "half": False, "thermo": 0, "every": 10,
         "steps": 20, "twojmax": 8},
        # A SNAP production box that fills the GPU, FP64.
        {"name": "snap_16k", "family": "driver", "pair": "snap", "nx": 20, "ny": 20, "nz": 20,
         "precision": "fp64", "neigh": "2D", "half": False, "thermo": 0, "every": 10,
         "steps": 10, "twojmax": 8},
        # A new configuration under a high-order potential (140 components).
        {"name": "snap_eval_2j12", "family": "eval", "nx": 8, "ny": 8, "nz": 8,
         "precision": "mixed", "twojmax": 12},
        # The ensemble benchmark: 256 uneven replicas, 256 to 6912 atoms each.
        {"name": "replicas_256", "family": "batch", "nrep": 256, "nmin": 256, "nmax": 8192,
         "sizes": 4, "precision": "mixed", "steps": 100},
        # Force-matching gradients: 64 SNAP configurations w.r.t. 56 coefficients, and 32 LJ
        # boxes w.r.t. (epsilon, sigma).
        {"name": "fit_snap_64", "family": "fit_snap", "count": 64, "smin": 4, "smax": 8,
         "precision": "fp64"},
        {"name": "fit_lj_32", "family": "fit_lj", "count": 32, "smin": 5, "smax": 10,
         "precision": "fp64"},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _box(rng, lo, hi):
    """three cell counts of a box whose mean edge is spread over lo..hi logarithmically"""
    n = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    return [max(int(lo), int(round(n * rng.uniform(0.8, 1.25)))) for _ in range(3)]


def draw(rng):
    kind = rng.choice(["driver_lj", "driver_lj", "driver_snap", "driver_snap", "modules", "eval",
                       "batch", "fit_snap", "fit_lj"])
    prec = rng.choice(["fp64", "mixed"])
    if kind == "driver_lj":
        nx, ny, nz = _box(rng, 5, 40)
        half = rng.random() < 0.25
        return {"family": "driver", "pair": "lj", "nx": nx, "ny": ny, "nz": nz,
                "precision": prec, "neigh": rng.choice(["2D", "CSR"]), "half": half,
                "thermo": rng.choice([0, 10]), "every": 20, "steps": rng.choice([20, 40, 60])}
    if kind == "driver_snap":
        nx, ny, nz = _box(rng, 4, 16)
        return {"family": "driver", "pair": "snap", "nx": nx, "ny": ny, "nz": nz,
                "precision": prec, "neigh": rng.choice(["2D", "CSR"]), "half": False,
                "thermo": rng.choice([0, 10]), "every": rng.choice([1, 10]), "steps": 10,
                "twojmax": rng.choice([6, 8, 8])}
    if kind == "modules":
        nx, ny, nz = _box(rng, 30, 80)
        return {"family": "modules", "nx": nx, "ny": ny, "nz": nz, "precision": prec,
                "neigh": rng.choice(["2D", "CSR"]), "every": 20, "steps": 20}
    if kind == "eval":
        nx, ny, nz = _box(rng, 4, 10)
        return {"family": "eval", "nx": nx, "ny": ny, "nz": nz, "precision": prec,
                "twojmax": rng.choice([6, 8, 10, 12])}
    if kind == "batch":
        nmin = _log_int(rng, 256, 1024)
        return {"family": "batch", "nrep": _log_int(rng, 8, 256), "nmin": nmin,
                "nmax": _log_int(rng, 2 * nmin, 8192), "sizes": rng.randrange(1000),
                "precision": prec, "steps": rng.choice([40, 70, 100])}
    smin = rng.randint(4, 6) if kind == "fit_snap" else rng.randint(5, 7)
    smax = smin + rng.randint(0, 2 if kind == "fit_snap" else 3)
    # fits are drawn in FP64: a few hundred values at most come back, sums of signed errors
    return {"family": kind, "count": _log_int(rng, 3, 48), "smin": smin, "smax": smax,
            "precision": "fp64"}


# ------------------------------------------------------------------ inputs
_FCC = np.array([(0, 0, 0), (0.5, 0.5, 0), (0.5, 0, 0.5), (0, 0.5, 0.5)])
_BCC = np.array([(0, 0, 0), (0.5, 0.5, 0.5)])


def _dev():
    return torch.device("cuda", 0)


def _gen(seed):
    g = torch.Generator(device=_dev())
    g.manual_seed(int(seed) * 7919 + 17)
    return g


def _lattice(case, basis, a):
    """sites cell by cell (z outermost, as the driver orders them) and the box"""
    nx, ny, nz = case["nx"], case["ny"], case["nz"]
    c = torch.cartesian_prod(*[torch.arange(k, device=_dev(), dtype=torch.float64)
                               for k in (nz, ny, nx)]).flip(1)
    b = torch.tensor(basis, device=_dev(), dtype=torch.float64)
    x = ((c[:, None, :] + b[None]) * a).reshape(-1, 3).contiguous()
    return x, (nx * a, ny * a, nz * a)


def _wrapped(x, box):
    L = torch.tensor(box, device=x.device, dtype=torch.float64)
    x = torch.where(x > L, x - L, x)
    return torch.where(x < 0, x + L, x)


def _atoms(case, seed, snap):
    """positions, velocities (device, FP64) and box of a case's seed"""
    g = _gen(seed)
    x, box = _lattice(case, _BCC if snap else _FCC, W_A if snap else LJ_A)
    # cut off at three standard deviations: no pair of the millions starts inside its core
    u = torch.randn(x.shape, generator=g, device=x.device, dtype=torch.float64)
    x = x + (0.1 if snap else 0.06) * u.clamp(-3.0, 3.0)
    v = torch.randn(x.shape, generator=g, device=x.device, dtype=torch.float64)
    v = v - v.mean(0)
    kT, m = (METAL_KB * W_T / METAL_MVV2E, W_MASS) if snap else (LJ_T, 1.0)
    v = v * math.sqrt(kT / m * (3 * len(v) - 3) / float((v * v).sum()))
    return _wrapped(x, box), v, box


def _beta(twojmax, seed=2024):
    return decks.snap_beta(seed=seed, sigma=0.05, ncoeff=len(flopcount.components(twojmax)))


# ----------------------------------------------------------- device arrays
class _Ptr:
    def __init__(self, ptr, shape, typestr):
        self.__cuda_array_interface__ = {"data": (ptr, False), "shape": shape,
                                         "typestr": typestr, "version": 2, "strides": None}


def _tensor(ptr, shape, typestr):
    """the library's device array as a tensor (no copy)"""
    return torch.as_tensor(_Ptr(C.cast(ptr, C.c_void_p).value, shape, typestr), device=_dev())


class _Out:
    """x, v, f of the local atoms in id order, gathered on the library's stream"""

    def __init__(self, ctx, n, mixed):
        L = emd.hip_lib()
        self.stream = torch.cuda.ExternalStream(L.emd_get_stream(ctx))
        self.mixed = mixed
        self.seen = {}
        opts = {"device": _dev(), "dtype": torch.float64}
        self.x, self.v = torch.empty((n, 3), **opts), torch.empty((n, 3), **opts)
        self.f = torch.empty((n, 3), device=_dev(),
                             dtype=torch.float32 if mixed else torch.float64)
        self.n = n
        self.at = torch.empty(n, device=_dev(), dtype=torch.int64)

    def _view(self, name, ptr, shape, typestr):
        key = C.cast(ptr, C.c_void_p).value
        if self.seen.get(name, (None,))[0] != key:
            self.seen[name] = (key, _tensor(ptr, shape, typestr))
        return self.seen[name][1]

    def take(self, s):
        n = self.n
        f = (self._view("f32", s.f32, (n, 3), "<f4") if self.mixed else
             self._view("f", s.f, (n, 3), "<f8"))
        with torch.cuda.stream(self.stream):
            torch.sub(self._view("id", s.id, (n,), "<i4"), 1, out=self.at)
            self.x.index_copy_(0, self.at, self._view("x", s.x, (n, 3), "<f8"))
            self.v.index_copy_(0, self.at, self._view("v", s.v, (n, 3), "<f8"))
            self.f.index_copy_(0, self.at, f)
        return {"x": self.x, "v": self.v, "f": self.f}


# ------------------------------------------------------------------ driver
def _restart_bytes(x, v):
    n = len(x)
    return b"".join([struct.pack("<i", n), np.arange(1, n + 1, dtype=np.int32).tobytes(),
                     np.zeros(n, np.int32).tobytes(), np.zeros(n).tobytes(),
                     np.ascontiguousarray(x).tobytes(), np.ascontiguousarray(v).tobytes(),
                     np.zeros((n, 3)).tobytes()])


def _lj_text(case):
    text = decks.lj_deck(n=1, steps=case["steps"], every=case["every"], thermo=case["thermo"],
                         newton=bool(case["half"]))
    return text.replace("block 0 1 0 1 0 1",
                        "block 0 %d 0 %d 0 %d" % (case["nx"], case["ny"], case["nz"]))


class _Driver:
    def __init__(self, case, seed):
        snap = case["pair"] == "snap"
        x, v, _ = _atoms(case, seed, snap)
        with tempfile.TemporaryDirectory() as d:
            path = os.path.join(d, "restart")
            with open(path, "wb") as f:
                f.write(_restart_bytes(x.cpu().numpy(), v.cpu().numpy()))
            if snap:
                coeff = decks.write(os.path.join(d, "W.snapcoeff"),
                                    decks.snap_coeff_text(_beta(case["twojmax"])))
                param = decks.write(os.path.join(d, "W.snapparam"), decks.SNAP_PARAM.replace(
                    "twojmax 8", "twojmax %d" % case["twojmax"]))
                text = decks.snap_deck(n=case["nx"], ny=case["ny"], nz=case["nz"],
                                       steps=case["steps"], every=case["every"],
                                       thermo=case["thermo"], coeff=coeff, param=param)
            else:
                text = _lj_text(case)
            deck = decks.write(os.path.join(d, "in.deck"), text)
            self.app = emd.App(
                ["-il", deck, "--restart", path, "--neigh-type", case["neigh"],
                 "--comm-type", "SERIAL", "--precision", case["precision"],
                 "--force-iteration", "NEIGH_HALF" if case["half"] else "NEIGH_FULL"]).init()
        self.app.set_phase_sync(False)
        self.steps = case["steps"]
        self.out = _Out(self.app.ctx, len(x), case["precision"] == "mixed")

    def run(self):
        self.app.run(self.steps)
        return self.out.take(self.app.L.emd_app_system(self.app.h).contents)


# ----------------------------------------------------------------- modules
def _i32(t):
    return C.c_void_p(t.data_ptr())


class _System:
    """an emd_system filled from device tensors, with its halo, bins and list"""

    def __init__(self, n, box, mass):
        self.ctx = emd.Context()
        self.L, self.h = self.ctx.L, self.ctx.h
        self.s, self.halo, self.bins, self.nl = EmdSystem(), EmdHalo(), EmdBins(), EmdNeigh()
        self.n, self.box = n, box
        self.types = torch.zeros(n, device=_dev(), dtype=torch.int32)
        self.ids = torch.arange(1, n + 1, device=_dev(), dtype=torch.int32)
        self.q = torch.zeros(n, device=_dev(), dtype=torch.float64)
        self.mass = (C.c_double * 1)(mass)
        self.have_mass = False

    def chk(self, status, what):
        self.ctx.check(status, what)

    def load(self, x, v):
        """the caller's device arrays into the system (stream-ordered copies)"""
        L, s = self.L, self.s
        view = lambda t: EmdVec3View(C.cast(C.c_void_p(t.data_ptr()), C.POINTER(C.c_double)),
                                     EMD_LAYOUT_RIGHT, 0)
        none = EmdVec3View(None, EMD_LAYOUT_RIGHT, 0)
        self.chk(L.emd_system_import(self.h, C.byref(s), self.n, view(x), view(v), none,
                                     _i32(self.types), _i32(self.ids), _i32(self.q)), "import")
        if not self.have_mass:
            self.chk(L.emd_system_set_mass(self.h, C.byref(s), 1, self.mass), "mass")
            self.have_mass = True
        s.n_local, s.n_ghost, s.n_global = self.n, 0, self.n
        for d in range(3):
            s.domain[d], s.lo[d], s.hi[d] = self.box[d], 0.0, self.box[d]

    def build(self, cut, newton, layout):
        L, h, s, b = self.L, self.h, C.byref(self.s), C.byref(self.bins)
        self.chk(L.emd_comm_exchange(h, s), "exchange")
        self.chk(L.emd_binning(h, s, cut, cut, cut, 1, 1, 0, 1, b), "bin sort")
        self.chk(L.emd_comm_exchange_halo(h, s, cut, C.byref(self.halo)), "halo")
        self.chk(L.emd_binning(h, s, cut, cut, cut, 1, 1, 1, 0, b), "bin")
        self.chk(L.emd_neigh_build(h, s, b, cut, 0, newton, layout, C.byref(self.nl)), "neigh")

    def __del__(self):
        try:
            self.L.emd_neigh_free(self.h, C.byref(self.nl))
            self.L.emd_bins_free(self.h, C.byref(self.bins))
            self.L.emd_halo_free(self.h, C.byref(self.halo))
            self.L.emd_system_free(self.h, C.byref(self.s))
        except Exception:
            pass


def _precision(case):
    return EMD_MIXED if case["precision"] == "mixed" else EMD_FP64


def _layout(case):
    return EMD_NEIGH_2D if case["neigh"] == "2D" else EMD_NEIGH_CSR


class _Modules:
    def __init__(self, case, seed):
        x, v, box = _atoms(case, seed, False)
        torch.cuda.synchronize()
        self.sys = _System(len(x), box, 1.0)
        self.prec, self.lay = _precision(case), _layout(case)
        self.steps, self.every = case["steps"], case["every"]
        self.p = EmdLJParams()
        self.p.ntypes = 1
        self.p.lj1[0][0], self.p.lj2[0][0], self.p.cutsq[0][0] = 48.0, 24.0, LJ_RC * LJ_RC
        self.sys.load(x, v)
        self.sys.build(LJ_RC + LJ_SKIN, 0, self.lay)
        self.force()
        self.out = _Out(self.sys.h, len(x), self.prec == EMD_MIXED)
        self.sys.ctx.sync()

    def force(self):
        y = self.sys
        y.chk(y.L.emd_lj_force_store(y.h, C.byref(y.s), C.byref(y.nl), C.byref(self.p),
                                     self.prec), "lj")

    def run(self):
        y, dtf, dtv, prec = self.sys, 0.5 * LJ_DT, LJ_DT, self.prec
        L, h, s, halo = y.L, y.h, C.byref(y.s), C.byref(y.halo)
        y.chk(L.emd_nve_initial(h, s, dtf, dtv, prec), "initial")
        for step in range(1, self.steps + 1):
            if step % self.every == 0:
                y.build(LJ_RC + LJ_SKIN, 0, self.lay)
            elif step == 1:
                y.chk(L.emd_comm_update_halo(h, s, halo), "update_halo")
            self.force()
            if step < self.steps:
                y.chk(L.emd_nve_step_boundary(h, s, halo, 0, int((step + 1) % self.every != 0),
                                              dtf, dtv, prec), "boundary")
        y.chk(L.emd_nve_final(h, s, dtf, prec), "final")
        return self.out.take(y.s)


# -------------------------------------------------------------------- eval
class _Eval:
    def __init__(self, case, seed):
        self.x, self.v, box = _atoms(case, seed, True)
        torch.cuda.synchronize()
        n = len(self.x)
        self.sys = _System(n, box, W_MASS)
        self.prec = _precision(case)
        self.beta = np.ascontiguousarray(_beta(case["twojmax"]))
        p = EmdSnapParams()
        p.twojmax, p.rfac0, p.rmin0, p.rcutfac = case["twojmax"], W_RFAC0, 0.0, W_RC
        p.switchflag, p.bzeroflag, p.radelem, p.wjelem = 1, 0, 0.5, 1.0
        p.ncoeff = len(self.beta) - 1
        p.coeff = self.beta.ctypes.data_as(C.POINTER(C.c_double))
        self.snap = C.c_void_p()
        self.sys.chk(self.sys.L.emd_snap_create(self.sys.h, C.byref(p), C.byref(self.snap)),
                     "snap_create")
        self.eatom = torch.zeros(n, device=_dev(), dtype=torch.float64)
        self.e = torch.zeros(n, device=_dev(), dtype=torch.float64)
        self.out = _Out(self.sys.h, n, self.prec == EMD_MIXED)
        torch.cuda.synchronize()

    def run(self):
        y, out = self.sys, self.out
        L, h, s, nl = y.L, y.h, C.byref(y.s), C.byref(y.nl)
        y.load(self.x, self.v)
        y.build(W_RC, 1, EMD_NEIGH_CSR)
        y.chk(L.emd_snap_force_zeroed(h, s, nl, self.snap, self.prec), "snap_force")
        y.chk(L.emd_comm_update_force(h, s, C.byref(y.halo), self.prec), "fold")
        total = C.c_double()
        y.chk(L.emd_snap_energy(h, s, nl, self.snap, C.byref(total),
                                C.cast(C.c_void_p(self.eatom.data_ptr()),
                                       C.POINTER(C.c_double))), "snap_energy")
        f = out.take(y.s)["f"]
        with torch.cuda.stream(out.stream):
            self.e.index_copy_(0, out.at, self.eatom)
        return {"f": f, "eatom": self.e, "energy": float(total.value)}

    def __del__(self):
        try:
            self.sys.L.emd_snap_destroy(self.sys.h, self.snap)
        except Exception:
            pass


# ------------------------------------------------------------------- batch
def _ensemble(case, seed):
    """replica sizes and densities from the case, positions and velocities from the seed"""
    shape = batch.ensemble(nrep=case["nrep"], seed=case["sizes"], nmin=case["nmin"],
                           nmax=case["nmax"])
    rng = np.random.default_rng(int(seed) * 31 + 5)
    n, L = shape["natoms"], np.repeat(shape["box"], shape["natoms"], axis=0)
    x = shape["x"] + rng.normal(0.0, 0.05, shape["x"].shape)
    x = np.where(x < 0, x + L, np.where(x > L, x - L, x))
    v = rng.normal(size=x.shape)
    start = np.concatenate([[0], np.cumsum(n)[:-1]])
    v -= np.repeat(np.add.reduceat(v, start, axis=0) / n[:, None], n, axis=0)
    t = np.add.reduceat((v * v).sum(1), start) / (3 * n - 3)
    v *= np.repeat(np.sqrt(shape["temp"] / t), n)[:, None]
    return n, shape["box"], x, v


class _Batch:
    def __init__(self, case, seed):
        n, box, x, v = _ensemble(case, seed)
        self.b = batch.Batch(n, box, precision=_precision(case))
        self.b.upload(x, v)
        self.b.setup()
        self.b.set_tile(8, 128)  # the tile the autotuner settles on for such an ensemble
        self.steps = case["steps"]

    def run(self):
        self.b.run(self.steps)
        ke, pe = self.b.thermo()
        x, v, f = self.b.download()
        return {"x": x, "v": v, "f": f, "ke": ke, "pe": pe}

    def __del__(self):
        try:
            self.b.close()
        except Exception:
            pass


# -------------------------------------------------------------------- fits
def _sizes(case):
    return tuple(range(case["smin"], case["smax"] + 1))


class _Fit:
    def __init__(self, case, seed):
        self.prec = _precision(case)
        if case["family"] == "fit_snap":
            true = forcematch.snap_beta_true(seed=2024)
            self.fm = forcematch.SnapForceMatchMerged(
                forcematch.snap_set(count=case["count"], seed=seed, sizes=_sizes(case)), true)
            self.theta = forcematch.snap_beta_perturbed(true, seed=seed + 1)
        else:
            self.fm = forcematch.LJForceMatchMerged(
                forcematch.lj_set(count=case["count"], seed=seed, sizes=_sizes(case)))
            self.theta = _lj_theta(seed)

    def run(self):
        loss, grad = self.fm.evaluate(self.theta, self.prec)
        return {"loss": loss, "grad": grad}

    def __del__(self):
        try:
            self.fm.close()
        except Exception:
            pass


def _lj_theta(seed):
    rng = np.random.default_rng(int(seed) + 2)
    return (1.0 + rng.normal(0.0, 0.05), 1.0 + rng.normal(0.0, 0.01))


_FAMILIES = {"driver": _Driver, "modules": _Modules, "eval": _Eval, "batch": _Batch,
             "fit_snap": _Fit, "fit_lj": _Fit}


def prepare(case, seed):
    return _FAMILIES[case["family"]](case, seed)


def run(state):
    return state.run()


# -------------------------------------------------------------------- work
def _lj_step(n, rows=1.0):
    """one LJ step: positions and velocities read and written, the list read; the distance of
    every listed pair and the force of every pair inside the cutoff"""
    per = 4.0 / 3.0 * math.pi * LJ_RHO
    listed_pairs, pairs = rows * per * (LJ_RC + LJ_SKIN) ** 3, rows * per * LJ_RC ** 3
    return n * (96.0 + 4.0 * listed_pairs), n * (9.0 * listed_pairs + 14.0 * pairs + 24.0)


def work(case):
    fam = case["family"]
    if fam == "batch":
        n = int(batch.ensemble(nrep=case["nrep"], seed=case["sizes"], nmin=case["nmin"],
                               nmax=case["nmax"])["natoms"].sum())
        b, f = _lj_step(n)
        return {"bytes": b * case["steps"], "flops": f * case["steps"]}
    if fam in ("fit_snap", "fit_lj"):
        sizes = _sizes(case)
        cells = sum(sizes[c % len(sizes)] ** 3 for c in range(case["count"]))
        if fam == "fit_lj":
            b, f = _lj_step(4 * cells)
            return {"bytes": b, "flops": 3.0 * f}
        # force and its adjoint: Y and F, W and S; U_tot of fixed configurations is known
        k = flopcount.snap_flops(8, 26)
        return {"bytes": 2.0 * cells * 16 * 285, "flops": 2.0 * cells * 2 * (k["Y"] + k["F"])}
    cells = case["nx"] * case["ny"] * case["nz"]
    if fam == "eval" or case.get("pair") == "snap":
        n, steps = 2 * cells, case.get("steps", 1)
        k = flopcount.snap_flops(case["twojmax"], 26)
        return {"bytes": n * steps * (96.0 + 4 * 58), "flops": n * steps * float(k["total"])}
    b, f = _lj_step(4 * cells, 0.5 if case.get("half") else 1.0)
    return {"bytes": b * case["steps"], "flops": f * case["steps"]}


# ------------------------------------------------- the same physics in torch
def _pairs(x, box, cut):
    """directed pairs (i, j) with |x_i - x_j| <= cut, nearest images (box edges at least twice
    the cutoff), from a padded cell table; all pairs where a box is under three cells wide"""
    n, dev = len(x), x.device
    L = torch.tensor(box, device=dev, dtype=torch.float64)
    nc = [int(b / cut) for b in box]
    got = []
    if min(nc) < 3:
        for i0 in range(0, n, 1024):
            d = x[i0:i0 + 1024, None, :] - x[None]
            d = d - L * torch.round(d / L)
            k = (d * d).sum(-1) <= cut * cut
            k[torch.arange(len(d), device=dev), torch.arange(i0, i0 + len(d), device=dev)] = False
            got.append(k.nonzero() + torch.tensor([i0, 0], device=dev))
        p = torch.cat(got)
        return p[:, 0].contiguous(), p[:, 1].contiguous()
    ncell = torch.tensor(nc, device=dev)
    c = (x / L * ncell).floor().long() % ncell
    flat = (c[:, 0] * nc[1] + c[:, 1]) * nc[2] + c[:, 2]
    order = torch.argsort(flat)
    count = torch.bincount(flat, minlength=nc[0] * nc[1] * nc[2])
    first = torch.cumsum(count, 0) - count
    most = int(count.max())
    table = torch.full((len(count), most), -1, device=dev, dtype=torch.int64)
    table[flat[order], torch.arange(n, device=dev) - first[flat[order]]] = order
    step = 1 << 20
    for i0 in range(0, n, step):
        xi, ci = x[i0:i0 + step], c[i0:i0 + step]
        for dx in (-1, 0, 1):
            for dy in (-1, 0, 1):
                for dz in (-1, 0, 1):
                    o = (ci + torch.tensor([dx, dy, dz], device=dev)) % ncell
                    j = table[(o[:, 0] * nc[1] + o[:, 1]) * nc[2] + o[:, 2]]
                    d = xi[:, None, :] - x[j.clamp(min=0)]
                    d -= L * torch.round(d / L)
                    k = (d * d).sum(-1) <= cut * cut
                    k &= (j >= 0) & (j != torch.arange(i0, i0 + len(xi), device=dev)[:, None])
                    r, s = k.nonzero(as_tuple=True)
                    got.append((r + i0, j[r, s]))
    return torch.cat([g[0] for g in got]), torch.cat([g[1] for g in got])


def _lj_forces(x, L, pi, pj, eps=1.0, sigma=1.0):
    """forces from directed pairs and, per atom, half of its pairs' shifted energies; L: box
    lengths, one row or one per atom"""
    f = torch.zeros_like(x)
    e = torch.zeros(len(x), device=x.device, dtype=torch.float64)
    lj1, lj2 = 48.0 * eps * sigma ** 12, 24.0 * eps * sigma ** 6
    c6 = LJ_RC ** -6
    for k in range(0, len(pi), 1 << 26):
        i, j = pi[k:k + (1 << 26)], pj[k:k + (1 << 26)]
        Li = L if L.dim() == 1 else L[i]
        d = x[i] - x[j]
        d -= Li * torch.round(d / Li)
        r2 = (d * d).sum(1)
        m = r2 < LJ_RC * LJ_RC
        i, d, r2 = i[m], d[m], 1.0 / r2[m]
        r6 = r2 ** 3
        f.index_add_(0, i, d * (r6 * (lj1 * r6 - lj2) * r2)[:, None])
        e.index_add_(0, i, (r6 * (0.5 * lj1 * r6 - lj2) - c6 * (0.5 * lj1 * c6 - lj2)) / 12.0)
    return f, e


def _md(x, v, box, steps, every, dt, dtf, cut, forces):
    """velocity Verlet with the list of the last rebuild, as a run of the driver"""
    pi, pj = _pairs(x, box, cut)
    f = forces(x, pi, pj)
    for step in range(1, steps + 1):
        v = v + dtf * f
        x = x + dt * v
        if step % every == 0:
            x = _wrapped(x, box)
            pi, pj = _pairs(x, box, cut)
        f = forces(x, pi, pj)
        v = v + dtf * f
    return x, v, f


# ---- SNAP: bispectrum components and their gradients by autograd
def _cg(j1, j2, j):
    """Clebsch-Gordan coefficients as a matrix [(j + 1), (j1 + 1)(j2 + 1)] (Racah's formula)"""
    F = math.factorial
    out = np.zeros((j + 1, j1 + 1, j2 + 1))
    for k1 in range(j1 + 1):
        for k2 in range(j2 + 1):
            a, b = 2 * k1 - j1, 2 * k2 - j2
            c = a + b
            if abs(c) > j:
                continue
            s = 0.0
            for z in range(max(0, -(j - j2 + a) // 2, -(j - j1 - b) // 2),
                           min((j1 + j2 - j) // 2, (j1 - a) // 2, (j2 + b) // 2) + 1):
                s += (-1.0) ** z / (F(z) * F((j1 + j2 - j) // 2 - z) * F((j1 - a) // 2 - z) *
                                    F((j2 + b) // 2 - z) * F((j - j2 + a) // 2 + z) *
                                    F((j - j1 - b) // 2 + z))
            d = math.sqrt(F((j1 + j2 - j) // 2) * F((j1 - j2 + j) // 2) * F((j2 - j1 + j) // 2) /
                          F((j1 + j2 + j) // 2 + 1))
            w = math.sqrt(F((j1 + a) // 2) * F((j1 - a) // 2) * F((j2 + b) // 2) *
                          F((j2 - b) // 2) * F((j + c) // 2) * F((j - c) // 2) * (j + 1))
            out[(c + j) // 2, k1, k2] = s * d * w
    return out.reshape(j + 1, -1)


class _Snap:
    def __init__(self, twojmax):
        self.J = twojmax
        self.comp = [(a, b, c) for a in range(twojmax + 1) for b in range(a + 1)
                     for c in range(a - b, min(twojmax, a + b) + 1, 2) if c >= a]
        self.cg = {t: torch.tensor(_cg(*t), device=_dev()) for t in self.comp}

    def layers(self, d, r, switched):
        """U_j of every pair times the switching function, layer by layer"""
        th = W_RFAC0 * math.pi * r / W_RC
        z0 = r / torch.tan(th)
        ri = torch.rsqrt(r * r + z0 * z0)
        ca = torch.complex(z0 * ri, d[:, 2] * ri)[:, None, None]        # conj(a)
        cb = torch.complex(d[:, 1] * ri, d[:, 0] * ri)[:, None, None]   # conj(b)
        sf = switched[:, None, None]
        u = torch.ones((len(r), 1, 1), device=r.device, dtype=torch.complex128)
        out = [u * sf]
        for j in range(1, self.J + 1):
            nb = j // 2 + 1
            ma = torch.arange(j + 1, device=r.device, dtype=torch.float64)[:, None]
            mb = torch.arange(nb, device=r.device, dtype=torch.float64)[None]
            rpa, rpb = torch.sqrt((j - ma) / (j - mb)), torch.sqrt(ma / (j - mb))
            prev = u[:, :, :nb]
            zero = torch.zeros((len(r), 1, prev.shape[2]), device=r.device, dtype=u.dtype)
            left = (rpa * ca * torch.cat([prev, zero], 1) - rpb * cb * torch.cat([zero, prev], 1))
            sign = 1.0 - 2.0 * ((ma + mb) % 2)
            right = (sign * left).conj().flip(1, 2)
            u = torch.cat([left, right[:, :, (1 if j % 2 == 0 else 0):]], 2)
            out.append(u * sf)
        return out

    def components(self, x, box, pi, pj, lo, hi):
        """B_k of atoms lo..hi - 1 and, per atom, the pair repulsion's energy (pairs sorted by
        i; box lengths one row or one per atom)"""
        a, b = (int(t) for t in torch.searchsorted(pi, torch.tensor([lo, hi], device=pi.device)))
        i, j = pi[a:b], pj[a:b]
        Li = box if box.dim() == 1 else box[i]
        d = x[j] - x[i]
        d = d - Li * torch.round(d.detach() / Li)
        m = (d.detach() ** 2).sum(1) < W_RC * W_RC
        i, d = i[m] - lo, d[m]
        r = torch.sqrt((d * d).sum(1))
        sf = 0.5 * (torch.cos(r * (math.pi / W_RC)) + 1.0)
        n = hi - lo
        U = []
        for jj, u in enumerate(self.layers(d, r, sf)):
            t = torch.eye(jj + 1, device=x.device, dtype=torch.complex128).expand(n, -1, -1)
            U.append(t.contiguous().index_add(0, i, u))
        B = []
        for t in self.comp:
            j1, j2, jj = t
            u1, u2, C1 = U[j1], U[j2], self.cg[t]
            p = u1[:, :, None, :, None] * u2[:, None, :, None, :]
            p = torch.view_as_real(p).permute(1, 2, 5, 0, 3, 4)
            k = (j1 + 1) * (j2 + 1)
            q = C1 @ p.reshape(k, -1)                       # ma | re im, n, mb1 mb2
            z = (q.reshape(-1, k) @ C1.t()).reshape(jj + 1, 2, n, jj + 1)
            w = torch.view_as_real(U[jj]).permute(1, 3, 0, 2)
            B.append((z * w).sum((0, 1, 3)))
        rep = torch.zeros(n, device=x.device, dtype=torch.float64).index_add(
            0, i, 1.25e5 * (r ** -12 - W_RC ** -12))
        return torch.stack(B, 1), rep

    def forces(self, x, box, pi, pj, beta, chunk):
        """forces and per-atom energies"""
        order = torch.argsort(pi, stable=True)
        pi, pj = pi[order], pj[order]
        f, es = torch.zeros_like(x), []
        for lo in range(0, len(x), chunk):
            hi = min(len(x), lo + chunk)
            y = x.detach().requires_grad_(True)
            B, rep = self.components(y, box, pi, pj, lo, hi)
            e = beta[0] + B @ beta[1:] + rep
            f -= torch.autograd.grad(e.sum(), y)[0]
            es.append(e.detach())
        return f, torch.cat(es)


def _exact_md(case, seed):
    snap = case.get("pair") == "snap"
    x, v, box = _atoms(case, seed, snap)
    L = torch.tensor(box, device=x.device, dtype=torch.float64)
    if snap:
        sn, beta = _Snap(case["twojmax"]), torch.tensor(_beta(case["twojmax"]), device=x.device)
        x, v, f = _md(x, v, box, case["steps"], case["every"], W_DT,
                      0.5 * W_DT / METAL_MVV2E / W_MASS, W_RC + W_SKIN,
                      lambda y, i, j: sn.forces(y, L, i, j, beta, 2048)[0])
    else:
        x, v, f = _md(x, v, box, case["steps"], case["every"], LJ_DT, 0.5 * LJ_DT,
                      LJ_RC + LJ_SKIN, lambda y, i, j: _lj_forces(y, L, i, j)[0])
    return {"x": x, "v": v, "f": f}


def _exact_eval(case, seed):
    x, _, box = _atoms(case, seed, True)
    L = torch.tensor(box, device=x.device, dtype=torch.float64)
    pi, pj = _pairs(x, box, W_RC)
    sn, beta = _Snap(case["twojmax"]), torch.tensor(_beta(case["twojmax"]), device=x.device)
    f, e = sn.forces(x, L, pi, pj, beta, 256 if case["twojmax"] > 8 else 2048)
    return {"f": f, "eatom": e, "energy": float(e.sum())}


def _exact_batch(case, seed):
    n, box, x, v = _ensemble(case, seed)
    x, v = (torch.tensor(t, device=_dev()) for t in (x, v))
    n_at = torch.tensor(n, device=_dev(), dtype=torch.int64)
    L = torch.repeat_interleave(torch.tensor(box, device=_dev()), n_at, dim=0)
    start = np.concatenate([[0], np.cumsum(n)])
    cut = LJ_RC + LJ_SKIN

    def wrap(y):
        y = torch.where(y > L, y - L, y)
        return torch.where(y < 0, y + L, y)

    def lists(y):
        got = [_pairs(y[start[r]:start[r + 1]], [float(b) for b in box[r]], cut)
               for r in range(len(n))]
        return tuple(torch.cat([g[k] + int(start[r]) for r, g in enumerate(got)]) for k in (0, 1))

    dt, x = LJ_DT, wrap(x)
    pi, pj = lists(x)
    f = _lj_forces(x, L, pi, pj)[0]
    for step in range(1, case["steps"] + 1):
        v = v + 0.5 * dt * f
        x = x + dt * v
        if step % 20 == 0:
            x = wrap(x)
            pi, pj = lists(x)
        f, e = _lj_forces(x, L, pi, pj)
        v = v + 0.5 * dt * f
    at = torch.repeat_interleave(torch.arange(len(n), device=_dev()), n_at)
    per = lambda t: torch.zeros(len(n), device=_dev(), dtype=torch.float64).index_add(0, at, t)
    return {"x": x, "v": v, "f": f, "ke": per(0.5 * (v * v).sum(1)), "pe": per(e)}


def _merged(configs, cut):
    """positions, box lengths per atom, pairs and first atom of every configuration"""
    xs, Ls, pis, pjs, start = [], [], [], [], [0]
    for x, box in configs:
        x = _wrapped(torch.tensor(x, device=_dev()), box)
        i, j = _pairs(x, box, cut)
        xs.append(x)
        Ls.append(torch.tensor(box, device=_dev(), dtype=torch.float64).expand(len(x), 3))
        pis.append(i + start[-1])
        pjs.append(j + start[-1])
        start.append(start[-1] + len(x))
    return torch.cat(xs), torch.cat(Ls), torch.cat(pis), torch.cat(pjs), start


def _exact_fit_snap(case, seed):
    true = forcematch.snap_beta_true(seed=2024)
    theta = forcematch.snap_beta_perturbed(true, seed=seed + 1)
    configs = forcematch.snap_set(count=case["count"], seed=seed, sizes=_sizes(case))
    sn, loss, grad = _Snap(8), 0.0, torch.zeros(len(true), device=_dev(), dtype=torch.float64)
    k = 0
    while k < len(configs):  # whole configurations, about two thousand atoms at a time
        m, n = k, 0
        while m < len(configs) and (m == k or n + len(configs[m][0]) <= 2048):
            n += len(configs[m][0])
            m += 1
        x, L, pi, pj, start = _merged(configs[k:m], W_RC)
        k = m
        order = torch.argsort(pi, stable=True)
        pi, pj = pi[order], pj[order]
        x = x.requires_grad_(True)
        db = torch.tensor(theta - true, device=_dev()).requires_grad_(True)
        B, _ = sn.components(x, L, pi, pj, 0, len(x))
        e = db[0] + B @ db[1:]
        df = -torch.autograd.grad(e.sum(), x, create_graph=True)[0]
        l = (df * df).sum()
        for a, b in zip(start, start[1:]):
            l = l + 100.0 * (e[a:b].sum() / (b - a)) ** 2
        grad += torch.autograd.grad(l, db)[0]
        loss += float(l.detach())
    return {"loss": loss, "grad": grad}


def _exact_fit_lj(case, seed):
    configs = forcematch.lj_set(count=case["count"], seed=seed, sizes=_sizes(case))
    x, L, pi, pj, start = _merged(configs, LJ_RC)
    d = x[pi] - x[pj]
    d = d - L[pi] * torch.round(d / L[pi])
    r2 = (d * d).sum(1)
    m = r2 < LJ_RC * LJ_RC
    pi, d, r2 = pi[m], d[m], 1.0 / r2[m]
    r6, c6 = r2 ** 3, LJ_RC ** -6

    def of(eps, sigma):
        s6 = sigma ** 6
        f = torch.zeros_like(x).index_add(
            0, pi, d * (r6 * (48.0 * eps * s6 * s6 * r6 - 24.0 * eps * s6) * r2)[:, None])
        pe = 2.0 * eps * (s6 * s6 * (r6 * r6 - c6 * c6) - s6 * (r6 - c6))
        return f, torch.zeros(len(x), device=_dev(), dtype=torch.float64).index_add(0, pi, pe)

    one = torch.ones((), device=_dev(), dtype=torch.float64)
    theta = [torch.tensor(t, device=_dev(), dtype=torch.float64, requires_grad=True)
             for t in _lj_theta(seed)]
    (f0, e0), (f1, e1) = of(one, one), of(*theta)
    loss = ((f1 - f0) ** 2).sum()
    for a, b in zip(start, start[1:]):
        loss = loss + 100.0 * ((e1[a:b] - e0[a:b]).sum() / (b - a)) ** 2
    grad = torch.stack(torch.autograd.grad(loss, theta))
    return {"loss": float(loss.detach()), "grad": grad}


_EXACT = {"driver": _exact_md, "modules": _exact_md, "eval": _exact_eval, "batch": _exact_batch,
          "fit_snap": _exact_fit_snap, "fit_lj": _exact_fit_lj}


def exact(case, seed):
    return _EXACT[case["family"]](case, seed)
