"""Plain and pruned batches on lists far from the origin against their spread,
where the split scan's error bound passes every probed row: the FP32 scan
serves them, in about the time of the same rows around the origin (the split
scan takes several times that), and lists that then move back to the origin
are split again.  Ids and distances of some queries against the oracle, of all
against the exact rescan's kernel (one query at a time)."""
import time

import numpy as np
import pytest

import oracle
from harmonyclient_amd import index as hx

pytestmark = pytest.mark.gpu


def _time(idx, q, n, k, P, algo):
    import torch
    D = torch.empty(n, k, device="cuda")
    I = torch.empty(n, k, dtype=torch.int64, device="cuda")
    prm = hx.make_params(nprobe=P, algo=algo)
    torch.cuda.synchronize()
    best = 1e9
    for _ in range(7):
        t = time.perf_counter()
        idx.search_device(n, q.data_ptr(), k, D.data_ptr(), I.data_ptr(), prm, stats=False)
        torch.cuda.synchronize()
        best = min(best, time.perf_counter() - t)
    return best, D.cpu().numpy(), I.cpu().numpy()


@pytest.mark.parametrize("metric,algo,offset", [(1, hx.ALGO_PLAIN, 1000.0), (1, hx.ALGO_PRUNED, 1000.0), (0, hx.ALGO_PLAIN, 1e5)])
@pytest.mark.parametrize("d", [64, 200])
def test_offset_lists(metric, algo, offset, d):
    import torch
    print(f"[case] metric={metric} algo={algo} d={d} offset={offset}", flush=True)
    rows, nlist, n, P, k = 100_000, 128, 1000, 32, 50
    r = np.random.default_rng(7)
    c = r.normal(0, 3, (nlist, d))
    xb0 = c[r.integers(0, nlist, rows)] + r.normal(0, 1, (rows, d))
    xq0 = c[r.integers(0, nlist, n)] + r.normal(0, 1, (n, d))
    idx = hx.Index(d, nlist, P, metric)
    times = {}
    for off in (0.0, offset, 0.0):
        xb, xq = (xb0 + off).astype(np.float32), (xq0 + off).astype(np.float32)
        cent = (c + off).astype(np.float32)
        if metric == 0:
            s = np.float32(np.linalg.norm(cent, axis=1).mean())
            xb, xq, cent = xb / s, xq / s, cent / s
        idx.set_centroids(cent)
        idx.add(rows, xb)
        times[off], D, I = _time(idx, torch.from_numpy(xq).cuda(), n, k, P, algo)
        ix = oracle.Index.build(metric, xb, cent)
        OD, OI, _ = ix.search(xq[:40], P, k)
        assert np.array_equal(I[:40], OI) and np.array_equal(D[:40].view(np.uint32), OD.view(np.uint32))
        for q in (100, 555, 999):
            D1, I1, _ = idx.search(1, xq[q:q + 1], k, params=hx.make_params(nprobe=P))
            assert np.array_equal(I1[0], I[q]) and np.array_equal(D1[0], D[q])
    print(f"[time] {times}", flush=True)
    if metric == 1:  # (of equal spread; an inner product's differs with the offset)
        assert times[offset] < 4.0 * times[0.0]
