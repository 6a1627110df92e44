"""emd_batch_download leaves the ensemble alone: the mixed forces are FP32
values, a second download gives the same, and a run continued after a download
(anywhere in a rebuild period, with and without graph replay) equals one that
never downloaded, bit for bit."""
import numpy as np
import pytest

import examinimd_amd as emd
from examinimd_amd import batch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", [emd.EMD_FP64, emd.EMD_MIXED])
@pytest.mark.parametrize("nrep,first,graph", [(1, 0, True), (1, 1, True), (3, 20, True),
                                              (3, 27, True), (5, 13, False)])
def test_download_leaves_the_run_alone(nrep, first, graph, prec):
    print(f"case: batch download, {nrep} replicas, after {first} steps, precision {prec}", flush=True)
    e = batch.ensemble(nrep=nrep, seed=nrep, nmin=256, nmax=1200)
    out = []
    for mid in (False, True):
        b = batch.Batch(e["natoms"], e["box"], precision=prec)
        b.upload(e["x"], e["v"])
        b.setup()
        b.run(first, graph=graph)
        if mid:
            d1, d2 = b.download(), b.download()
            for p, q in zip(d1, d2):
                assert np.array_equal(p, q)
            assert np.abs(d1[2]).max() > 0.0
            if prec == emd.EMD_MIXED:
                assert np.array_equal(d1[2], d1[2].astype(np.float32).astype(np.float64))
        b.run(33, graph=graph)
        out.append(b.download() + b.thermo())
        b.close()
    for p, q in zip(*out):
        assert np.array_equal(p, q)
