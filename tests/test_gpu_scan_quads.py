"""The per-query scan at every remainder of its eight quads at a time, whole rows and
pruning blocks, rows with a partial last quad: against the oracle."""
import numpy as np
import pytest

import oracle
from harmonyclient_amd import index as hx

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("metric", [0, 1])
@pytest.mark.parametrize("d", [1, 4, 7, 9, 16, 20, 24, 28, 31, 32, 36, 43, 48, 60, 75, 92, 124, 225, 300])
def test_remainders(d, metric):
    print(f"[case] d={d} metric={metric}", flush=True)
    r = np.random.default_rng(d)
    xb = r.normal(0, 1, (700, d)).astype(np.float32)
    cent = xb[:6].copy()
    idx = hx.Index(d, 6, 1, metric)
    idx.set_centroids(cent)
    idx.add(700, xb)
    ix = oracle.Index.build(metric, xb, cent)
    xq = r.normal(0, 1, (5, d)).astype(np.float32)
    OD, OI, _ = ix.search(xq, 4, 13)
    _, pr = idx.coarse(xq, 4)
    for prm in (dict(),) if metric == 0 else (dict(), dict(algo=hx.ALGO_PRUNED), dict(algo=hx.ALGO_PRUNED, dim_block=5),
                                              dict(algo=hx.ALGO_PRUNED, dim_block=28)):
        D, I, _ = idx.scan(xq, pr, 13, **prm)
        assert np.array_equal(I, OI) and np.array_equal(D.view(np.uint32), OD.view(np.uint32)), prm
    tau = idx.warmup_tau(xq, pr, 13, L=2, W=70)
    assert np.array_equal(tau.view(np.uint32), ix.warmup_tau(xq, pr, 13, 2, 70).view(np.uint32))
