"""SNAP forces and the adjoint's W at the edges of the lane groups: a
wavefront takes seven neighbours (nine lanes each) up to twojmax 8 and four
(thirteen lanes) up to 12, a block of the force kernel four wavefronts.  Clusters
whose atoms have 1 to 33 neighbours, the smallest, odd and even layers.
Forces against the oracle with those of zero coefficients taken off (the pair
repulsion of a tight cluster is far larger), the adjoint as the transpose of
that force.  About 1e5 products per component in two orders, of terms up to a
few hundred times the result: 1e-10 of the largest force, and 1e-14 of the
largest repulsion that was taken off; 1e-4 in mixed precision."""
import numpy as np
import pytest

import examinimd_amd as emd
from examinimd_amd import decks

pytestmark = pytest.mark.gpu
RC = 4.73442


def cluster(n, rng):
    """n points in a ball of radius RC / 2 (every pair a neighbour), the
    distances as even as a draw of 200 candidates each makes them"""
    x = np.zeros((1, 3))
    while len(x) < n:
        c = rng.normal(size=(200, 3))
        c *= (2.3 * rng.random((200, 1)) ** (1 / 3)) / np.linalg.norm(c, axis=1)[:, None]
        d = np.linalg.norm(c[:, None] - x[None], axis=2).min(1)
        x = np.vstack([x, c[d.argmax()]])
    return x + 8.0


@pytest.mark.parametrize("twojmax", [0, 1, 3, 8, 9, 12])
@pytest.mark.parametrize("n", [2, 4, 5, 7, 8, 9, 17, 18, 29, 30, 34])
def test_force_and_adjoint_at_group_edges(oracle, n, twojmax):
    from examinimd_amd.pipeline import Pipeline
    from test_oracle import _energy_force
    print(f"case: SNAP cluster of {n} atoms, twojmax {twojmax}", flush=True)
    rng = np.random.default_rng(100 * n + twojmax)
    x, box = cluster(n, rng), 16.0
    nc = oracle.lib().or_snap_ncoeff(twojmax)
    beta = np.array(decks.snap_beta(seed=3, sigma=0.05, ncoeff=nc))
    zero = np.zeros(nc + 1)

    def ref(b):
        return _energy_force(oracle, x, box, "snap", cut=RC + 1.0,
                             snap=oracle.snap_params(list(b), twojmax=twojmax))[1]

    F0 = ref(zero)
    want = ref(beta) - F0
    pl = Pipeline()
    pl.load(x, (box,) * 3, mass=183.84)
    pl.build(RC + 1.0, newton=1)
    pl.snap_setup(list(zero), twojmax=twojmax)
    z = {p: pl.snap_force(p) for p in (emd.EMD_FP64, emd.EMD_MIXED)}
    pl.snap_set_coeff(beta)
    got = {p: pl.snap_force(p) - z[p] for p in z}
    g = rng.normal(size=(n, 3))
    adj = pl.snap_adjoint(g, 0.0, emd.EMD_FP64)
    pl.close()
    top, rep = np.abs(want).max(), np.abs(F0).max()
    e64 = np.abs(got[emd.EMD_FP64] - want).max()
    e32 = np.abs(got[emd.EMD_MIXED] - want).max()
    print("force", top, "repulsion", rep, "errors", e64, e32)
    assert e64 <= 1e-10 * top + 1e-14 * rep
    assert e32 <= 1e-4 * top + 1e-6 * rep
    ea = abs(adj @ beta - (g * want).sum())
    assert ea <= 1e-10 * np.abs(g).sum() * top + 1e-14 * rep * np.abs(g).sum()
