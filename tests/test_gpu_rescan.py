"""The exact rescan of queries that overflow their survivor buffer, one query
split over several workgroups or many over one each, against the oracle: list
lengths around the edges of the split, k from 1 to the largest, more parts
than tiles, rows with equal distances.  Ids and distances bit for bit."""
import numpy as np
import pytest

import oracle
from harmonyclient_amd import index as hx

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows,d,nlist,n,P,k", [
    (20000, 20, 8, 1, 8, 100), (20000, 20, 8, 2, 8, 1024), (3000, 70, 8, 7, 8, 1), (3000, 70, 30, 64, 30, 17),
    (3000, 8, 8, 511, 3, 40), (3000, 8, 8, 512, 3, 40), (3000, 8, 8, 513, 3, 40), (3000, 8, 8, 1100, 3, 40),
    (2000, 420, 300, 5, 300, 64), (300, 3, 4, 3, 1, 200),
])
@pytest.mark.parametrize("data", ["int", "real", "dup"])
def test_rescan(rows, d, nlist, n, P, k, data):
    print(f"[case] {data} {rows} x {d} nlist={nlist} n={n} P={P} k={k}", flush=True)
    r = np.random.default_rng(rows + n)
    xb, xq = (r.normal(0, 40, (m, d)) + 100 for m in (rows, n))
    if data == "int":
        xb, xq = (np.clip(np.rint(x), 0, 255) for x in (xb, xq))
    elif data == "dup":
        xb = np.rint(xb[r.integers(0, 3, rows)])
    xb, xq = xb.astype(np.float32), xq.astype(np.float32)
    cent = xb[r.permutation(rows)[:nlist]].copy()
    ix = oracle.Index.build(1, xb, cent)
    idx = hx.Index(d, nlist, 1, 1)
    idx.set_centroids(cent)
    idx.add(rows, xb)
    OD, OI, _ = ix.search(xq, P, k)
    D, I, st = idx.search(n, xq, k, params=hx.make_params(nprobe=P, algo=hx.ALGO_BATCHED, tau=hx.TAU_NONE, survivor_cap=2))
    assert st.fallback_queries > 0
    assert np.array_equal(I, OI), f"{(I != OI).sum()} ids differ"
    assert np.array_equal(D.view(np.uint32), OD.view(np.uint32))
