"""emd_lj_force_energy_store against the two calls it replaces (bit for bit),
and emd_fit_residual against numpy on the downloaded forces and energies: a
difference and a doubling per component (exact, so equal bits), sums of
squares and of per-atom energies in another order (1e-13 of the sum of the
absolute terms, ~4000 terms)."""
import ctypes as C

import numpy as np
import pytest

import examinimd_amd as emd
from examinimd_amd import forcematch as fm
from examinimd_amd.abi import EmdLJParams
from examinimd_amd.pipeline import Pipeline, lattice

pytestmark = pytest.mark.gpu


def _put(pl, a):
    p = C.c_void_p()
    pl.chk(pl.L.emd_malloc(pl.ctx.h, C.byref(p), max(a.nbytes, 8)), "malloc")
    pl.chk(pl.L.emd_memcpy_h2d(pl.ctx.h, p, a.ctypes.data_as(C.c_void_p), a.nbytes), "h2d")
    return p


def _get(pl, p, n):
    out = np.zeros(n)
    pl.chk(pl.L.emd_memcpy_d2h(pl.ctx.h, out.ctypes.data_as(C.c_void_p), p, out.nbytes), "d2h")
    return out


@pytest.mark.parametrize("prec", [emd.EMD_FP64, emd.EMD_MIXED])
@pytest.mark.parametrize("n,cuts", [(1, [0, 1]), (85, [0, 85]), (86, [0, 1, 1, 86]),
                                    (257, []), (1372, [0, 300, 556, 1372])])
def test_residuals_and_energies(n, cuts, prec):
    print(f"case: fit residual, {n} atoms, configurations {cuts}, precision {prec}", flush=True)
    rng = np.random.default_rng(n)
    x = (lattice("fcc", 7, 1.68) + rng.normal(0, 0.04, (1372, 3)))[:n]
    pl = Pipeline()
    pl.load(x, (7 * 1.68,) * 3)
    pl.build(2.5)
    L, c, s, nl = pl.L, pl.ctx.h, C.byref(pl.s), C.byref(pl.nl)
    p = EmdLJParams()
    p.ntypes = 1
    p.lj1[0][0], p.lj2[0][0], p.cutsq[0][0] = 48.0, 24.0, 6.25
    d = lambda q: C.cast(q, C.POINTER(C.c_double))
    e1, e2 = _put(pl, np.zeros(n)), _put(pl, np.zeros(n))
    pl.chk(L.emd_lj_force_store(c, s, nl, C.byref(p), prec), "force")
    pl.chk(L.emd_lj_energy_atoms(c, s, nl, C.byref(p), 0, d(e1)), "energy")
    want = pl.forces(prec)
    pl.chk(L.emd_force_zero(c, s, prec), "zero")
    pl.chk(L.emd_lj_force_energy_store(c, s, nl, C.byref(p), prec, d(e2)), "both")
    assert np.array_equal(pl.forces(prec), want)
    eat = _get(pl, e1, n)
    assert np.array_equal(_get(pl, e2, n), eat)

    F = want[pl._device_ids() - 1]
    ft = F + rng.normal(0, 0.5, F.shape)
    nconf = max(0, len(cuts) - 1)
    start = np.array(cuts if nconf else [0], np.int32)
    E = np.array([eat[a:b].sum() for a, b in zip(cuts, cuts[1:])])
    et = E + rng.normal(0, 3.0, nconf)
    g, w = _put(pl, np.zeros(3 * n)), _put(pl, np.zeros(n))
    pl.chk(L.emd_fit_residual(c, s, prec, d(_put(pl, ft)), d(g), nconf,
                              C.cast(_put(pl, start), C.POINTER(C.c_int)), d(e1),
                              d(_put(pl, et if nconf else np.zeros(1))), d(w), None), "residual")
    loss = C.c_double()
    pl.chk(L.emd_fit_loss(c, C.byref(loss)), "loss")
    assert np.array_equal(_get(pl, g, 3 * n).reshape(n, 3), 2.0 * (F - ft))
    ref = ((F - ft) ** 2).sum()
    got_w = _get(pl, w, n)
    for k in range(nconf):
        a, b = cuts[k], cuts[k + 1]
        if b > a:
            de = E[k] - et[k]
            ref += 100.0 * (de / (b - a)) ** 2
            tol = 1e-13 * (np.abs(eat[a:b]).sum() + abs(et[k]))
            assert np.abs(got_w[a:b] - 200.0 * de / (b - a) ** 2).max() <= 200.0 * tol / (b - a) ** 2
    assert abs(loss.value - ref) <= 1e-12 * ref
    pl.close()


@pytest.mark.parametrize("prec", [emd.EMD_FP64, emd.EMD_MIXED])
@pytest.mark.parametrize("layout", [emd.EMD_NEIGH_CSR, emd.EMD_NEIGH_2D])
@pytest.mark.parametrize("ntypes,table,lanes", [(1, True, 0), (2, False, 0), (2, True, 0),
                                                (20, True, 0), (2, False, 1), (1, False, 8),
                                                (2, False, 16)])
def test_forces_and_energies_of_several_types(ntypes, table, lanes, layout, prec):
    """emd_lj_force_energy_store with per-pair coefficients and cutoffs (the
    fixed arrays, a table, more types than the arrays hold) and with other lane
    counts: the bits of emd_lj_force_store and emd_lj_energy_atoms"""
    print(f"case: force and energy, {ntypes} types, table {table}, lanes {lanes}, layout {layout}, "
          f"precision {prec}", flush=True)
    rng = np.random.default_rng(ntypes)
    n = 1371
    x = (lattice("fcc", 7, 1.68) + rng.normal(0, 0.04, (1372, 3)))[:n]
    types = rng.integers(0, ntypes, n)
    types[0] = ntypes - 1
    sig = rng.uniform(0.9, 1.05, (ntypes, ntypes))
    eps, rc = rng.uniform(0.5, 1.5, (ntypes, ntypes)), rng.uniform(1.5, 2.5, (ntypes, ntypes))
    coeff = np.array([48.0 * eps * sig ** 12, 24.0 * eps * sig ** 6, rc * rc])
    coeff = np.ascontiguousarray(0.5 * (coeff + coeff.transpose(0, 2, 1)))
    p = EmdLJParams()
    p.ntypes = ntypes
    if table:
        p.table = coeff.ctypes.data_as(C.POINTER(C.c_double))
    else:
        for a in range(ntypes):
            for b in range(ntypes):
                p.lj1[a][b], p.lj2[a][b], p.cutsq[a][b] = (float(k) for k in coeff[:, a, b])
    pl = Pipeline()
    pl.load(x, (7 * 1.68,) * 3, types=types)
    pl.build(2.5, layout=layout)
    L, c, s, nl = pl.L, pl.ctx.h, C.byref(pl.s), C.byref(pl.nl)
    if lanes:
        pl.chk(L.emd_lj_set_lanes(c, prec, lanes), "lanes")
    d = lambda q: C.cast(q, C.POINTER(C.c_double))
    e1, e2 = _put(pl, np.zeros(n)), _put(pl, np.ones(n))
    pl.chk(L.emd_lj_force_store(c, s, nl, C.byref(p), prec), "force")
    pl.chk(L.emd_lj_energy_atoms(c, s, nl, C.byref(p), 0, d(e1)), "energy")
    want = pl.forces(prec)
    pl.chk(L.emd_force_zero(c, s, prec), "zero")
    pl.chk(L.emd_lj_force_energy_store(c, s, nl, C.byref(p), prec, d(e2)), "both")
    got, eat, both = pl.forces(prec), _get(pl, e1, n), _get(pl, e2, n)
    pl.close()
    assert np.abs(want).max() > 1.0 and np.abs(eat).max() > 1.0
    assert np.array_equal(got, want)
    assert np.array_equal(both, eat)


def test_targets_can_be_replaced():
    """the merged sets keep their targets on the device: assigning other ones
    changes the loss as the definition says"""
    s = fm.LJForceMatchMerged(fm.lj_set(count=2))
    l0, _ = s.evaluate((1.0, 1.0), emd.EMD_FP64, grad=False)
    assert l0 == 0.0
    s.Ft = s.Ft + 1.0
    s.Et = s.Et + 2.0
    l1, _ = s.evaluate((1.0, 1.0), emd.EMD_FP64, grad=False)
    n = s.m.n_atoms
    want = 3.0 * n.sum() + 100.0 * ((2.0 / n) ** 2).sum()
    assert abs(l1 - want) <= 1e-9 * want
    s.close()


def _loss(s, theta):
    return s.evaluate(theta, emd.EMD_FP64, grad=False)[0]


@pytest.mark.parametrize("kind", ["lj", "snap"])
def test_targets_changed_in_place(kind):
    """changes of elements of the target arrays count in the next evaluation,
    before the first read and after it, as do later changes in an array that
    was assigned; the arrays outlive close()"""
    print(f"case: targets changed in place, {kind}", flush=True)
    if kind == "lj":
        s, theta = fm.LJForceMatchMerged(fm.lj_set(count=2)), (1.0, 1.0)
    else:
        theta = fm.snap_beta_true(seed=5)
        s = fm.SnapForceMatchMerged(fm.snap_set(count=2, seed=3, sizes=(4,)), theta)
    n = s.m.n_atoms
    base = _loss(s, theta)  # 0, or (the fold's atomic order) rounding
    assert base <= 1e-15
    s.Ft[3] += (1.0, 2.0, 0.0)
    s.Ft[-1, 2] -= 1.5
    want = 1.0 + 4.0 + 2.25
    assert abs(_loss(s, theta) - want) <= 1e-9 * want
    s.Et[1] += 3.0
    want += 100.0 * (3.0 / n[1]) ** 2
    assert abs(_loss(s, theta) - want) <= 1e-9 * want
    F = s.Ft.copy()
    s.Ft = F
    F[0, 0] += 0.5
    want += 0.25
    assert abs(_loss(s, theta) - want) <= 1e-9 * want
    s.close()
    assert np.array_equal(s.Ft, F)


def test_targets_of_other_shapes():
    """a target broadcasts to its shape, a wrong one raises before anything is
    copied to the device"""
    print("case: targets of other shapes", flush=True)
    s = fm.LJForceMatchMerged(fm.lj_set(count=3))
    n, F, E = s.m.n_atoms, s.Ft.copy(), s.Et.copy()
    s.Et = 0.0
    want = 100.0 * ((E / n) ** 2).sum()
    assert abs(_loss(s, (1.0, 1.0)) - want) <= 1e-9 * want
    s.Et, s.Ft = E, [0.0, 0.0, 0.0]
    want = (F ** 2).sum()
    assert abs(_loss(s, (1.0, 1.0)) - want) <= 1e-9 * want
    for wrong in (np.zeros((len(F) + 1, 3)), np.zeros((len(F) - 1, 3)), np.zeros(3 * len(F))):
        s.Ft = wrong
        with pytest.raises(ValueError):
            _loss(s, (1.0, 1.0))
    s.Ft = F
    for wrong in (np.zeros(2), np.zeros(4)):
        s.Et = wrong
        with pytest.raises(ValueError):
            _loss(s, (1.0, 1.0))
    s.Et = list(E)
    assert _loss(s, (1.0, 1.0)) == 0.0
    s.close()
