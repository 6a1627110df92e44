"""emd_comm_update_force with one launch per dimension (both faces' ghosts at
once; per phase where an atom owns a ghost on either face, in boxes thinner
than twice the halo) against the sequential fold f[pack_p] += f[ghosts_p],
p = 5..0, bit for bit."""
import ctypes as C

import numpy as np
import pytest

import examinimd_amd as emd
from examinimd_amd.pipeline import Pipeline, lattice

pytestmark = pytest.mark.gpu
A_W = 3.1803


@pytest.mark.parametrize("prec", [emd.EMD_FP64, emd.EMD_MIXED])
@pytest.mark.parametrize("nc,cut,wide", [(2, 5.73442, 1), (3, 5.73442, 1), (4, 5.73442, 1),
                                         (7, 5.73442, 1), (3, 5.73442, 16)])
def test_fold_per_dimension(monkeypatch, nc, cut, wide, prec):
    print(f"case: fold per dimension, BCC {nc}^3 x {wide}, cut {cut}, precision {prec}",
          flush=True)
    monkeypatch.setenv("EMD_FOLD_ONE", "0")
    x = lattice("bcc", nc, A_W)
    x = np.concatenate([x + (0, k * nc * A_W, 0) for k in range(wide)])  # thin in x and z only
    x += np.random.default_rng(nc).normal(0, 0.05, x.shape)
    dt = np.float32 if prec == emd.EMD_MIXED else np.float64
    pl = Pipeline()
    pl.load(x, (nc * A_W, wide * nc * A_W, nc * A_W), mass=183.84)
    pl.build(cut, newton=1)
    L, c = pl.L, pl.ctx.h
    n, counts = pl.s.n_local, [pl.h.num_ghost[p] for p in range(6)]
    packs = []
    for p in range(6):
        arr = np.zeros(counts[p], np.int32)
        pl.chk(L.emd_memcpy_d2h(c, arr.ctypes.data_as(C.c_void_p),
                                C.cast(pl.h.pack[p], C.c_void_p), arr.nbytes), "pack")
        packs.append(arr)
    f = np.random.default_rng(7).normal(0, 1, (n + sum(counts), 3)).astype(dt)
    dst = pl.s.f32 if prec == emd.EMD_MIXED else pl.s.f
    pl.chk(L.emd_memcpy_h2d(c, C.cast(dst, C.c_void_p), f.ctypes.data_as(C.c_void_p), f.nbytes), "f")
    pl.chk(L.emd_comm_update_force(c, C.byref(pl.s), C.byref(pl.h), prec), "fold")
    got = np.zeros((n, 3), dt)
    pl.chk(L.emd_memcpy_d2h(c, got.ctypes.data_as(C.c_void_p), C.cast(dst, C.c_void_p),
                            got.nbytes), "download")
    pl.close()
    want = f.copy()
    off = n + np.concatenate([[0], np.cumsum(counts)])
    for p in range(5, -1, -1):
        want[packs[p]] += want[off[p]:off[p] + counts[p]]
    assert sum(counts) > 0
    thin = [len(np.intersect1d(packs[p], packs[p + 1])) > 0 for p in (0, 2, 4)]
    assert thin == [edge < 2 * cut for edge in (nc * A_W, wide * nc * A_W, nc * A_W)]
    print("thin", thin, "differ", int((got != want[:n]).sum()))
    assert np.array_equal(got, want[:n])
