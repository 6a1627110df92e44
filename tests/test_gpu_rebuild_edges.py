"""Binning and CSR row offsets at the edges of their kernels: one workgroup
(7168 atoms, 4096 bins) against the counting sort above it, bins holding more
atoms than a wavefront, and the row scan in one workgroup (32 768 rows)
against three launches.  The expected permutation is numpy's stable sort by
bin id, with the bin arithmetic of BinOp3D as emd_binning documents it
(src/binning_types/binning_kksort.cpp:71-125); whole numbers, no tolerance."""
import ctypes as C

import numpy as np
import pytest

import examinimd_amd as emd
from examinimd_amd.pipeline import Pipeline

pytestmark = pytest.mark.gpu


def bin_ids(x, b):
    n = np.array([b.nbinx, b.nbiny, b.nbinz])
    lo = np.array([b.minx, b.miny, b.minz])
    hi = np.array([b.maxx, b.maxy, b.maxz])
    k = ((1.0 * n / (hi - lo)) * (x - lo)).astype(np.int64)
    return (k[:, 0] * n[1] + k[:, 1]) * n[2] + k[:, 2]


@pytest.mark.parametrize("n,edge,cut,cluster", [
    (1, 9.0, 2.8, 0), (64, 9.0, 2.8, 0), (1025, 12.0, 2.8, 0), (1500, 12.0, 2.8, 1500),
    (7168, 14.0, 1.0, 0), (7168, 14.1, 1.0, 200), (7169, 14.0, 1.0, 0), (9000, 20.0, 2.8, 300),
    (9000, 60.0, 2.8, 64), (9000, 60.0, 2.8, 65), (9000, 60.0, 2.8, 256), (9000, 60.0, 2.8, 257)])
def test_binning_permutation(n, edge, cut, cluster):
    print(f"case: binning {n} atoms, bins {cut} in {edge}, cluster {cluster}", flush=True)
    rng = np.random.default_rng(n + cluster)
    x = rng.uniform(0.0, edge, (n, 3))
    if cluster:
        x[rng.choice(n, cluster, replace=False)] = rng.uniform(0.4, 0.6, (cluster, 3)) * cut
    pl = Pipeline()
    pl.load(x, (edge,) * 3)
    L, c, s, b = pl.L, pl.ctx.h, C.byref(pl.s), pl.b
    pl.chk(L.emd_binning(c, s, cut, cut, cut, 1, 1, 0, 0, C.byref(b)), "bin")
    ids = bin_ids(x, b)
    count = np.bincount(ids, minlength=b.nbins)
    assert np.array_equal(emd.download_ints(c, b.bincount, b.nbins), count)
    assert np.array_equal(emd.download_ints(c, b.binoffsets, b.nbins), np.cumsum(count) - count)
    assert np.array_equal(emd.download_ints(c, b.permute, n), np.argsort(ids, kind="stable"))
    assert b.max_count == count.max()
    pl.close()


@pytest.mark.parametrize("n", [1, 4097, 32768, 32769])
def test_csr_offsets_and_total(n):
    print(f"case: CSR offsets of {n} rows", flush=True)
    edge = max(9.0, (n / 0.3) ** (1.0 / 3.0))
    x = np.random.default_rng(n).uniform(0.0, edge, (n, 3))
    pl = Pipeline()
    pl.load(x, (edge,) * 3)
    for again in range(2):  # counted and filled, then one pass into the known capacity
        pl.build(1.5)
        num = emd.download_ints(pl.ctx.h, pl.nl.num, n)
        row = emd.download_ints(pl.ctx.h, pl.nl.row, n + 1)
        assert np.array_equal(row, np.concatenate([[0], np.cumsum(num)]))
        assert pl.nl.total == num.sum() and pl.nl.maxneighs == num.max()
    pl.close()


@pytest.mark.parametrize("n", [864, 6000, 40000])
def test_arrays_are_complete_with_their_counts(n):
    """a call that returns a count has waited for the arrays that go with it
    (the stream is idle where nothing is queued behind the count: binning
    without sort, exchange_halo, a padded list of known width); with
    emd_set_early_counts it need not have, and the arrays are the same"""
    import torch
    print(f"case: arrays complete with their counts, {n} atoms", flush=True)
    edge, cut = (n / 0.8) ** (1.0 / 3.0), 1.5
    pl = Pipeline()
    pl.load(np.random.default_rng(n).uniform(0.0, edge, (n, 3)), (edge,) * 3)
    L, c, s, h, b = pl.L, pl.ctx.h, C.byref(pl.s), pl.h, pl.b
    for again in range(2):
        pl.build(cut, layout=emd.EMD_NEIGH_2D)  # capacities
    stream = torch.cuda.ExternalStream(L.emd_get_stream(c))
    got = []
    for early in (0, 1):
        if early:
            was = C.c_int(-1)
            pl.chk(L.emd_set_early_counts(c, 1, C.byref(was)), "early counts")
            assert was.value == 0
        idle, out = [], []

        def took(*arrays):
            idle.append(stream.query())
            out.extend(emd.download_ints(c, ptr, k) for ptr, k in arrays)

        pl.chk(L.emd_binning(c, s, cut, cut, cut, 1, 1, 0, 0, C.byref(b)), "bin")
        took((b.permute, n), (b.bincount, b.nbins), (b.binoffsets, b.nbins))
        pl.chk(L.emd_comm_exchange_halo(c, s, cut, C.byref(h)), "halo")
        ng = pl.s.n_ghost
        took((h.root, ng), (h.image, ng), (pl.s.id, n + ng),
             *[(h.pack[p], h.num_ghost[p]) for p in range(6)])
        pl.chk(L.emd_binning(c, s, cut, cut, cut, 1, 1, 1, 0, C.byref(b)), "bin all")
        took((b.permute, n + ng), (b.bincount, b.nbins), (b.binoffsets, b.nbins))
        pl.chk(L.emd_neigh_build(c, s, C.byref(b), cut, 0, 0, emd.EMD_NEIGH_2D,
                                 C.byref(pl.nl)), "neigh")
        took((pl.nl.num, n))
        num = out[-1]
        ent = emd.download_ints(c, pl.nl.entries, n * pl.nl.maxneighs).reshape(n, -1)
        out.append(ent[np.arange(ent.shape[1]) < num[:, None]])
        print("early", early, "idle after each call", idle)
        if not early:
            assert all(idle)
        got.append(out)
    pl.close()
    assert all(np.array_equal(p, q) for p, q in zip(*got)) and len(got[0]) == len(got[1])
