"""Learned-bound searches whose model predicts far above every distance: the
lists' radii bound the prediction, results are those of the oracle.  k at the
edges of 32-row tiles, above the nearest list's rows and above all probed rows;
integer and real lists; probe counts per query; a hidden width of the fused
inference and one past it.  Ids and distances bit for bit."""
import numpy as np
import pytest
import torch

import oracle
from harmonyclient_amd import index as hx

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("k", [1, 32, 33, 100, 400, 1024])
@pytest.mark.parametrize("data,hidden,per_query", [("int", 128, False), ("int", 72, True), ("int", 144, False), ("real", 128, True)])
def test_prediction_above_the_radii(data, hidden, per_query, k):
    print(f"[case] {data} hidden={hidden} npq={per_query} k={k}", flush=True)
    rows, d, nlist, n, P = 4000, 24, 40, 150, 12
    r = np.random.default_rng(k + hidden)
    centres = r.uniform(0, 255, (nlist, d))
    xb, xq = (centres[r.integers(0, nlist, m)] + r.normal(0, 6, (m, d)) for m in (rows, n))
    if data == "int":
        xb, xq = (np.clip(np.rint(x), 0, 255) for x in (xb, xq))
    xb, xq = xb.astype(np.float32), xq.astype(np.float32)
    cent = centres.astype(np.float32)
    ix = oracle.Index.build(1, xb, cent)
    idx = hx.Index(d, nlist, P, 1)
    idx.set_centroids(cent)
    idx.add(rows, xb)
    m = hx.TauModel(hidden=hidden)
    f = hx.N_FEATURES
    p = np.zeros(f * hidden + hidden * hidden + 3 * hidden + 1 + 2 * f + 2, np.float32)
    p[f * hidden + hidden * hidden + 3 * hidden] = 60.0  # b3: tau = expm1(60)
    p[-2 - f:-2] = 1.0
    p[-2] = 1.0
    m.set_params(p)
    idx.set_tau_model(m)
    counts = r.integers(1, P + 1, n).astype(np.int32) if per_query else np.full(n, P, np.int32)
    dev = torch.from_numpy(counts).cuda()
    prm = hx.make_params(nprobe=P, algo=hx.ALGO_BATCHED, tau=hx.TAU_LEARNED,
                         nprobe_per_query_dev=dev.data_ptr() if per_query else None)
    D, I, st = idx.search(n, xq, k, params=prm)
    for c in np.unique(counts):
        at = np.flatnonzero(counts == c)
        OD, OI, _ = ix.search(xq[at], int(c), k)
        assert np.array_equal(I[at], OI), f"{(I[at] != OI).sum()} ids differ"
        assert np.array_equal(D[at].view(np.uint32), OD.view(np.uint32))
    assert st.overflow_queries == 0
    if k <= 33 and not per_query:  # without the radii every probed row survives
        assert st.survivors < 0.7 * n * P * rows / nlist
