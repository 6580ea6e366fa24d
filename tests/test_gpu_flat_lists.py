"""Plain and pruned batches where the planning counts with atomics (past 4096 and
8192 lists) and where the split scan prepares its own queries (one probe):
against the oracle, device calls without statistics (the split scan) and host
calls with them."""
import numpy as np
import pytest

import oracle
from harmonyclient_amd import index as hx

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("metric", [1, 0])
@pytest.mark.parametrize("rows,d,nlist,n,P,k", [
    (40_000, 24, 4500, 1500, 120, 12), (40_000, 24, 9000, 1500, 200, 12),
    (60_000, 33, 8, 3000, 1, 20), (60_000, 130, 8, 2000, 1, 20),
])
def test_many_lists_and_one_probe(rows, d, nlist, n, P, k, metric):
    import torch
    print(f"[case] rows={rows} d={d} nlist={nlist} n={n} P={P} metric={metric}", flush=True)
    r = np.random.default_rng(nlist)
    c = r.normal(0, 3, (min(nlist, 200), d))
    xb, xq = ((c[r.integers(0, len(c), m)] + r.normal(0, 1, (m, d))).astype(np.float32) for m in (rows, n))
    cent = xb[:nlist].copy()
    idx = hx.Index(d, nlist, P, metric)
    idx.set_centroids(cent)
    idx.add(rows, xb)
    m = 60
    OD, OI, _ = oracle.Index.build(metric, xb, cent).search(xq[-m:], P, k)
    q = torch.from_numpy(xq).cuda()
    for algo in (hx.ALGO_PLAIN, hx.ALGO_PRUNED)[:1 + metric]:
        prm = hx.make_params(nprobe=P, algo=algo)
        D = torch.empty(n, k, device="cuda")
        I = torch.empty(n, k, dtype=torch.int64, device="cuda")
        torch.cuda.synchronize()
        idx.search_device(n, q.data_ptr(), k, D.data_ptr(), I.data_ptr(), prm, stats=False)
        torch.cuda.synchronize()
        D, I = D.cpu().numpy(), I.cpu().numpy()
        assert np.array_equal(I[-m:], OI) and np.array_equal(D[-m:].view(np.uint32), OD.view(np.uint32))
        Dh, Ih, _ = idx.search(n, xq, k, params=prm)
        assert np.array_equal(I, Ih) and np.array_equal(D, Dh)
