"""Per-atom SNAP energies, formed as a third of Re(conj(U) Y), against
beta_0 + sum_k beta_k B_k + repulsion from emd_snap_descriptors (which sums
every component's Z products): the smallest systems (fewer atoms than a block
has wavefronts, isolated atoms), odd and even twojmax of both size classes,
bzeroflag on and off.  The two add the same ~4e4 (4e5) products in different
orders: 1e-11 of the sum of |beta_k B_k|."""
import ctypes as C

import numpy as np
import pytest

import examinimd_amd as emd
from examinimd_amd import decks, flopcount
from examinimd_amd.pipeline import Pipeline, lattice

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("bzero", [0, 1])
@pytest.mark.parametrize("twojmax", [0, 1, 3, 8, 9, 12])
@pytest.mark.parametrize("n", [1, 2, 5, 54])
def test_energy_equals_descriptor_sum(n, twojmax, bzero):
    print(f"case: SNAP energy, {n} atoms, twojmax {twojmax}, bzero {bzero}", flush=True)
    rng = np.random.default_rng(10 * n + twojmax)
    x = (lattice("bcc", 3, 3.2) + rng.normal(0, 0.1, (54, 3)))[:n]
    if n == 5:
        x[4] = (9.0, 9.0, 9.0)
    nc = len(flopcount.components(twojmax))
    beta = decks.snap_beta(seed=7, sigma=0.05, ncoeff=nc, beta0=0.3)
    pl = Pipeline()
    pl.load(x, (13.0,) * 3, mass=183.84)
    pl.build(4.73442, newton=1)
    pl.snap_setup(list(beta), twojmax=twojmax, bzeroflag=bzero)
    L, c = pl.L, pl.ctx.h

    def dev(count):
        p = C.c_void_p()
        pl.chk(L.emd_malloc(c, C.byref(p), 8 * count), "malloc")
        return p, C.cast(p, C.POINTER(C.c_double))

    def host(p, count):
        out = np.zeros(count)
        pl.chk(L.emd_memcpy_d2h(c, out.ctypes.data_as(C.c_void_p), p, out.nbytes), "d2h")
        return out

    (pb, db), (pe, de) = dev(n * nc), dev(n)
    pl.chk(L.emd_snap_descriptors(c, C.byref(pl.s), C.byref(pl.nl), pl.snap, db), "descriptors")
    B = host(pb, n * nc).reshape(n, nc)
    total = C.c_double()
    pl.chk(L.emd_snap_energy(c, C.byref(pl.s), C.byref(pl.nl), pl.snap, C.byref(total), de), "e")
    e = host(pe, n)
    xs = np.zeros(3 * n)
    pl.chk(L.emd_system_download(c, C.byref(pl.s), n, xs.ctypes.data_as(C.POINTER(C.c_double)),
                                 None, None, None, None, None), "x")
    d = xs.reshape(n, 1, 3) - xs.reshape(1, n, 3)
    d -= 13.0 * np.round(d / 13.0)
    r2 = (d * d).sum(2) + 1e9 * np.eye(n)
    rep = np.where(r2 < 4.73442 ** 2, 1.25e5 * (r2 ** -6 - 4.73442 ** -12), 0.0).sum(1)
    want = beta[0] + B @ beta[1:] + rep
    scale = np.abs(B) @ np.abs(beta[1:]) + np.abs(rep) + 1.0
    print("largest difference", np.abs(e - want).max(), "scale", scale.max())
    assert (np.abs(e - want) <= 1e-11 * scale).all()
    assert abs(total.value - e.sum()) <= 1e-12 * np.abs(e).sum()
    pl.close()


@pytest.mark.parametrize("twojmax", [4, 8])
def test_energy_is_of_the_present_positions_with_static_geometry(twojmax):
    """emd_snap_static_geometry keeps geometry for force and adjoint calls
    only: an energy after the atoms have moved is bit for bit that of a SNAP
    object that kept nothing, and it drops what was kept, so the force after it
    is that object's too (atomic additions in another order: 1e-12 of the largest)"""
    print(f"case: SNAP energy, static geometry, moved atoms, twojmax {twojmax}", flush=True)
    n, a = 128, 3.1803
    rng = np.random.default_rng(twojmax)
    x = lattice("bcc", 4, a) + rng.normal(0, 0.05, (n, 3))
    beta = list(decks.snap_beta(seed=7, sigma=0.05, ncoeff=len(flopcount.components(twojmax))))
    pl, fresh = Pipeline(), None
    try:
        pl.load(x, (4 * a,) * 3, mass=183.84)
        pl.build(5.73442, newton=1)
        pl.snap_setup(beta, twojmax=twojmax)
        L, c = pl.L, pl.ctx.h
        pl.chk(L.emd_snap_static_geometry(c, pl.snap, 1), "static")
        fresh = Pipeline(pl.ctx)
        fresh.snap_setup(beta, twojmax=twojmax)
        kept, new = pl.snap, fresh.snap
        first = [pl.snap_energy(), pl.snap_force(emd.EMD_FP64)]
        xs = np.zeros(3 * n)
        pl.chk(L.emd_memcpy_d2h(c, xs.ctypes.data_as(C.c_void_p), C.cast(pl.s.x, C.c_void_p),
                                xs.nbytes), "d2h")
        xs += rng.normal(0, 0.05, 3 * n)
        pl.chk(L.emd_memcpy_h2d(c, C.cast(pl.s.x, C.c_void_p), xs.ctypes.data_as(C.c_void_p),
                                xs.nbytes), "h2d")
        pl.chk(L.emd_comm_update_halo(c, C.byref(pl.s), C.byref(pl.h)), "halo")
        got = [pl.snap_energy(), pl.snap_force(emd.EMD_FP64)]
        pl.snap = new
        want = [pl.snap_energy(), pl.snap_force(emd.EMD_FP64)]
        pl.snap = kept
    finally:
        if fresh is not None:
            fresh.close()
        pl.close()
    assert got[0] == want[0] != first[0]
    scale = np.abs(want[1]).max()
    assert np.abs(got[1] - want[1]).max() <= 1e-12 * scale < np.abs(first[1] - want[1]).max()
