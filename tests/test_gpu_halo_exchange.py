"""exchange_halo against the six phases written out in numpy
(CommSerial::exchange_halo, src/comm_types/comm_serial.cpp:55-97 and
comm_serial.h:112-181): phase counts, pack lists, owners, image codes and
every ghost's data, bit for bit, at the edges of the kernels' tiles (a
wavefront of 64 atoms, a block of 1024, one workgroup's 2048) and in a box
thinner than twice the halo depth, where an atom has both images of a
dimension.  Position copies and one addition per shifted dimension: no
tolerance."""
import ctypes as C

import numpy as np
import pytest

import examinimd_amd as emd
from examinimd_amd.pipeline import Pipeline

pytestmark = pytest.mark.gpu


def six_phases(x, box, depth):
    """(x with ghosts, pack list per phase, owner and image code per ghost)"""
    n = len(x)
    xs, root, image, packs = x.copy(), [], [], []
    owner, code = np.arange(n), np.zeros(n, np.int64)
    last = 0
    for phase in range(6):
        d, hi = phase // 2, phase % 2 == 0
        cand = len(xs) - (0 if hi else last)
        c = xs[:cand, d]
        src = np.nonzero(c >= box[d] - depth if hi else c <= 0.0 + depth)[0]
        new = xs[src].copy()
        new[:, d] += -box[d] if hi else box[d]
        owner = np.concatenate([owner, owner[src]])
        code = np.concatenate([code, code[src] | ((1 if hi else 2) << (2 * d))])
        xs = np.concatenate([xs, new])
        packs.append(src)
        last = len(src)
    return xs, packs, owner[n:], code[n:]


@pytest.mark.parametrize("one", ["1", "0"])
@pytest.mark.parametrize("n,box,depth", [
    (1, (9.0, 9.0, 9.0), 2.8), (63, (9.0, 9.0, 9.0), 2.8), (65, (9.0, 11.0, 13.0), 2.8),
    (1025, (4.0, 15.0, 12.0), 2.8), (2048, (14.0, 13.0, 14.0), 2.8),
    (2049, (14.0, 13.0, 14.0), 2.8), (20001, (30.0, 28.0, 29.0), 2.8)])
def test_exchange_halo_equals_six_phases(monkeypatch, n, box, depth, one):
    print(f"case: exchange_halo of {n} atoms, box {box}, one workgroup {one}", flush=True)
    monkeypatch.setenv("EMD_HALO_ONE", one)
    rng = np.random.default_rng(n)
    x = rng.uniform(0.0, 1.0, (n, 3)) * box
    x[:: 7, 0] = 0.0                       # on a face
    x[3:: 11, 1] = box[1] - depth          # on a threshold
    v = rng.normal(size=x.shape)
    types = rng.integers(0, 3, n)
    types[0] = 2
    pl = Pipeline()
    pl.load(x, box, v=v, types=types)
    L, c, s = pl.L, pl.ctx.h, C.byref(pl.s)
    want, packs, owner, code = six_phases(x, np.array(box), depth)
    for again in range(2):  # the second call has the capacities of the first
        pl.chk(L.emd_comm_exchange_halo(c, s, depth, C.byref(pl.h)), "halo")
        ng = len(owner)
        assert [pl.h.num_ghost[p] for p in range(6)] == [len(p) for p in packs]
        assert pl.s.n_ghost == pl.h.n_ghost == ng
        for p in range(6):
            assert np.array_equal(emd.download_ints(c, pl.h.pack[p], len(packs[p])), packs[p])
        assert np.array_equal(emd.download_ints(c, pl.h.root, ng), owner)
        assert np.array_equal(emd.download_ints(c, pl.h.image, ng), code)
        tot = n + ng
        xs, vs, qs = np.zeros((tot, 3)), np.zeros((tot, 3)), np.full(tot, np.nan)
        ts, ids = np.zeros(tot, np.int32), np.zeros(tot, np.int32)
        P = lambda a, t: a.ctypes.data_as(C.POINTER(t))
        pl.chk(L.emd_system_download(c, s, tot, P(xs, C.c_double), P(vs, C.c_double), None,
                                     P(ts, C.c_int), P(ids, C.c_int), P(qs, C.c_double)), "d2h")
        who = np.concatenate([np.arange(n), owner])
        assert np.array_equal(xs, want)
        assert np.array_equal(vs, v[who])
        assert np.array_equal(ts, types[who])
        assert np.array_equal(ids, who + 1)
        assert np.array_equal(qs, np.zeros(tot))
    pl.close()
