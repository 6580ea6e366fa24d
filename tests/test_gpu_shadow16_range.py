"""Batched searches of real-valued lists whose components are all of about the
largest magnitude (dense positive data, a common offset): the queries' norms
exceed what a component of the FP16 shadow may, none of their components does,
and no query is handed to the exact rescans.  One whose components do leave
FP16's range is, and only it.  Ids and distances against the oracle."""
import numpy as np
import pytest

import oracle
from harmonyclient_amd import index as hx

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("d", [64, 100, 128, 129, 420])
@pytest.mark.parametrize("n", [40, 3200])
@pytest.mark.parametrize("kind", ["uniform", "offset"])
def test_dense_queries_stay_in_range(d, n, kind):
    print(f"[case] {kind} d={d} n={n}", flush=True)
    rows, nlist, P, k = 4000, 20, 6, 10
    r = np.random.default_rng(d)

    def data(m):
        return (r.uniform(0, 1, (m, d)) if kind == "uniform" else 8.0 + r.normal(0, 1, (m, d))).astype(np.float32)

    xb, xq = data(rows), data(n)
    xq[3] *= np.float32(1e3)  # its components leave FP16 at the lists' scale
    cent = xb[:nlist].copy()
    idx = hx.Index(d, nlist, P, 1)
    idx.set_centroids(cent)
    idx.add(rows, xb)
    D, I, st = idx.search(n, xq, k, params=hx.make_params(nprobe=P, algo=hx.ALGO_BATCHED))
    m = 64
    OD, OI, _ = oracle.Index.build(1, xb, cent).search(xq[:m], P, k)
    assert np.array_equal(I[:m], OI) and np.array_equal(D[:m].view(np.uint32), OD.view(np.uint32))
    assert st.scan_kind == 0 and st.fallback_queries == 1
