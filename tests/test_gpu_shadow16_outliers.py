"""Batched searches of real-valued lists with a few components far above the
rest: the shadow's error bound must stay one that most rows fail (FP16's
absolute part grows with the largest value, BF16's bound does not), whatever
the largest value.  Ids and distances against the oracle."""
import numpy as np
import pytest

import oracle
from harmonyclient_amd import index as hx

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("d", [24, 200])
@pytest.mark.parametrize("outlier", [0.0, 1e3, 1e5, 1e6, 1e7, 1e8, 1e13])
@pytest.mark.parametrize("zeros", [False, True])
def test_one_large_component(d, outlier, zeros):
    print(f"[case] d={d} outlier={outlier} zeros={zeros}", flush=True)
    rows, nlist, n, P, k = 12000, 30, 200, 30, 10
    r = np.random.default_rng(3)
    c = r.normal(0, 4, (nlist, d))

    def data(m):
        return (c[r.integers(0, nlist, m)] + r.normal(0, 1, (m, d))).astype(np.float32)

    xb, xq = data(rows), data(n)
    if zeros:
        xb[::5] = 0.0
    cent = xb[1:nlist + 1].copy()
    if outlier:
        xb[777, 5] = outlier
    idx = hx.Index(d, nlist, P, 1)
    idx.set_centroids(cent)
    idx.add(rows, xb)
    OD, OI, _ = oracle.Index.build(1, xb, cent).search(xq, P, k)
    D, I, st = idx.search(n, xq, k, params=hx.make_params(nprobe=P, algo=hx.ALGO_BATCHED))
    assert np.array_equal(I, OI) and np.array_equal(D.view(np.uint32), OD.view(np.uint32))
    # (a query's own component is 1/30 of the rows; the zero rows are a list's worth more)
    assert st.fallback_queries == 0 and st.survivors < st.candidates // 4, (st.survivors, st.candidates)
