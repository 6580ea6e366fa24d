"""Pruned batches with their own warm-up lists and rows: the results do not
depend on them, and a few lists of many rows cost no more than the default
(they are not taken as that many rows of ten lists)."""
import time

import numpy as np
import pytest

import oracle
from harmonyclient_amd import index as hx

pytestmark = pytest.mark.gpu


def test_warmup_of_one_long_list():
    import torch
    print("[case] pruned, 5000 queries, warm-up forms", flush=True)
    r = np.random.default_rng(4)
    rows, d, nlist, n, P, k = 300_000, 128, 512, 5000, 32, 20
    c = r.uniform(0, 255, (nlist, d))

    def data(m):
        return np.clip(np.rint(c[r.integers(0, nlist, m)] + r.normal(0, 20, (m, d))), 0, 255).astype(np.float32)

    xb, xq = data(rows), data(n)
    cent = np.rint(c).astype(np.float32)
    idx = hx.Index(d, nlist, P, 1)
    idx.set_centroids(cent)
    idx.add(rows, xb)
    OD, OI, _ = oracle.Index.build(1, xb, cent).search(xq[-20:], P, k)
    q = torch.from_numpy(xq).cuda()
    D = torch.empty(n, k, device="cuda")
    I = torch.empty(n, k, dtype=torch.int64, device="cuda")
    ms = {}
    for L, W in ((10, 0), (1, 5000), (1, 1), (32, 64), (2, 300), (0, 0), (300, 7)):
        prm = hx.make_params(nprobe=P, algo=hx.ALGO_PRUNED, warmup_lists=L, warmup_list_size=W)
        t = []
        for _ in range(7):
            torch.cuda.synchronize()
            t0 = time.perf_counter()
            idx.search_device(n, q.data_ptr(), k, D.data_ptr(), I.data_ptr(), prm, stats=False)
            torch.cuda.synchronize()
            t.append((time.perf_counter() - t0) * 1e3)
        ms[L, W] = min(t)
        assert np.array_equal(I[-20:].cpu().numpy(), OI) and np.array_equal(D[-20:].cpu().numpy(), OD)
    print(f"[time] {ms}", flush=True)
    assert ms[1, 5000] < 1.5 * ms[10, 0]
