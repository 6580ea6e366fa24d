"""Planning at the (query, probe) counts where its workgroups change size, with
and without radius classes, and in chunks whose last is smaller; a sample of
the queries against the oracle.  Ids and distances bit for bit."""
import numpy as np
import pytest

import oracle
from harmonyclient_amd import index as hx

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("algo,n,P", [
    (hx.ALGO_BATCHED, 1024, 1), (hx.ALGO_BATCHED, 1025, 1), (hx.ALGO_BATCHED, 8192, 16), (hx.ALGO_BATCHED, 8193, 16),
    (hx.ALGO_BATCHED, 16384, 16), (hx.ALGO_BATCHED, 16385, 16), (hx.ALGO_PLAIN, 4096, 32), (hx.ALGO_PLAIN, 4097, 32),
    (hx.ALGO_PLAIN, 8500, 32),
])
@pytest.mark.parametrize("nlist", [40, 1100])
def test_plan_sizes(algo, n, P, nlist):
    print(f"[case] algo={algo} n={n} P={P} nlist={nlist}", flush=True)
    rows, d, k = 30000, 12, 10
    r = np.random.default_rng(n + nlist)
    xb, xq = (np.clip(np.rint(r.normal(0, 40, (m, d)) + 100), 0, 255).astype(np.float32) for m in (rows, n))
    cent = xb[r.permutation(rows)[:nlist]].copy()
    ix = oracle.Index.build(1, xb, cent)
    idx = hx.Index(d, nlist, P, 1)
    idx.set_centroids(cent)
    idx.add(rows, xb)
    D, I, _ = idx.search(n, xq, k, params=hx.make_params(nprobe=P, algo=algo))
    at = np.unique(np.concatenate([np.arange(8), np.arange(n - 8, n), r.integers(0, n, 48)]))
    OD, OI, _ = ix.search(xq[at], P, k)
    assert np.array_equal(I[at], OI), f"{(I[at] != OI).sum()} ids differ"
    assert np.array_equal(D[at].view(np.uint32), OD.view(np.uint32))
