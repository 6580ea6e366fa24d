"""The workgroup scan of the FP16 shadow (real lists past 128 dims) against the
oracle: chunk counts around its groups of four, queries per list around its
items' 32 and 64, lists around its tile pairs and items, queries that FP16
cannot hold beside ordinary ones.  Ids and distances bit for bit."""
import numpy as np
import pytest

import oracle
from harmonyclient_amd import index as hx

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("d", [129, 144, 176, 192, 209, 256, 385, 512])
@pytest.mark.parametrize("rows,nlist,n,P", [(700, 6, 31, 6), (1100, 3, 33, 3), (2100, 2, 64, 2), (1300, 9, 65, 5), (40, 3, 129, 3),
                                            (5000, 70, 200, 40)])
@pytest.mark.parametrize("huge", [False, True])
def test_shadow_wg(d, rows, nlist, n, P, huge):
    print(f"[case] {rows} x {d} nlist={nlist} n={n} P={P} huge={huge}", flush=True)
    r = np.random.default_rng(d + rows)
    c = r.normal(0, 3, (nlist, d))
    xb, xq = ((c[r.integers(0, nlist, m)] + r.standard_t(3.0, (m, d))).astype(np.float32) for m in (rows, n))
    if huge:
        xq[0] *= 1e9
        xq[n // 2] *= 1e9
    cent = xb[r.permutation(rows)[:nlist]].copy()
    ix = oracle.Index.build(1, xb, cent)
    idx = hx.Index(d, nlist, P, 1)
    idx.set_centroids(cent)
    idx.add(rows, xb)
    OD, OI, _ = ix.search(xq, P, 10)
    D, I, st = idx.search(n, xq, 10, params=hx.make_params(nprobe=P, algo=hx.ALGO_BATCHED))
    assert st.batch_queries == 64
    assert np.array_equal(I, OI), f"{(I != OI).sum()} ids differ"
    assert np.array_equal(D.view(np.uint32), OD.view(np.uint32))
