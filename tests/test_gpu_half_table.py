"""The half-list force kernel adds a block's forces up in an LDS table of 1024
slots before they go to memory.  Cases where the table overflows (unrelated
atoms consecutive in memory, every neighbour of a block different, rows far
longer than usual), where it collides and where a block is partly empty,
against the full-list kernel on the same positions.  Both sum the same pair
forces (~50-250 of them, |F| up to ~1e3) in another order: 1e-12 of the
largest force in FP64; mixed rounds each of those sums to FP32, 1e-5."""
import ctypes as C

import numpy as np
import pytest

import examinimd_amd as emd
from examinimd_amd.abi import EmdLJParams, EmdNeigh
from examinimd_amd.pipeline import Pipeline

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", [emd.EMD_FP64, emd.EMD_MIXED])
@pytest.mark.parametrize("n,rho,shuffle", [(1, 0.1, False), (33, 0.3, False), (4000, 0.8, False),
                                           (4000, 0.8, True), (3001, 3.0, True)])
def test_half_forces_equal_full_forces(n, rho, shuffle, prec):
    print(f"case: half-list LJ table, {n} atoms at {rho}, shuffled {shuffle}, {prec}", flush=True)
    rng = np.random.default_rng(n)
    k = int(np.ceil(n ** (1.0 / 3.0)))
    g = np.stack(np.meshgrid(*[np.arange(k)] * 3, indexing="ij"), -1).reshape(-1, 3)[:n]
    a = rho ** (-1.0 / 3.0)
    edge = max(k * a, 6.0)
    x = (g + 0.5 + rng.uniform(-0.1, 0.1, (n, 3))) * (edge / k)
    if shuffle:
        x = x[rng.permutation(n)]
    sigma = 0.9 * min(1.0, edge / k)
    pl = Pipeline()
    pl.load(x, (edge,) * 3)
    L, c, s = pl.L, pl.ctx.h, C.byref(pl.s)
    # without the sorting pass atoms stay in the caller's order
    pl.chk(L.emd_comm_exchange_halo(c, s, 2.8, C.byref(pl.h)), "halo")
    pl.chk(L.emd_binning(c, s, 2.8, 2.8, 2.8, 1, 1, 1, 0, C.byref(pl.b)), "bin")
    p = EmdLJParams()
    p.ntypes = 1
    p.lj1[0][0], p.lj2[0][0], p.cutsq[0][0] = 48.0 * sigma ** 12, 24.0 * sigma ** 6, 6.25
    out = []
    for half in (0, 1):
        nl = EmdNeigh()
        pl.chk(L.emd_neigh_build(c, s, C.byref(pl.b), 2.8, half, 1, emd.EMD_NEIGH_CSR,
                                 C.byref(nl)), "neigh")
        pl.chk(L.emd_force_zero(c, s, prec), "zero")
        pl.chk(L.emd_lj_force(c, s, C.byref(nl), C.byref(p), prec, half), "lj")
        if half:
            pl.chk(L.emd_comm_update_force(c, s, C.byref(pl.h), prec), "fold")
        out.append(pl.forces(prec))
        pl.chk(L.emd_neigh_free(c, C.byref(nl)), "free")
    scale = np.abs(out[0]).max() if n > 1 else 1.0
    err = np.abs(out[1] - out[0]).max()
    print("largest force", scale, "difference", err)
    assert err <= (1e-12 if prec == emd.EMD_FP64 else 1e-5) * max(scale, 1e-300)
    pl.close()
