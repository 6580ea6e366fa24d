"""Host searches whose batches grow from call to call: the pinned buffers that
queries and results go through are not made anew on every call, so a first pass
over growing sizes takes little more than a second one.  (The device buffers
are at their size before, by a device search of the largest batch.)"""
import time

import numpy as np
import pytest

from harmonyclient_amd import index as hx

pytestmark = pytest.mark.gpu


def test_growing_batches():
    import torch
    print("[case] host searches of 1, 8, 15, ... 1499 queries, twice", flush=True)
    d, nlist, k, n = 128, 64, 10, 1500
    r = np.random.default_rng(1)
    xb = np.clip(np.rint(r.normal(128, 40, (20_000, d))), 0, 255).astype(np.float32)
    xq = np.clip(np.rint(r.normal(128, 40, (n, d))), 0, 255).astype(np.float32)
    ratios = []
    for _ in range(3):
        idx = hx.Index(d, nlist, 1, 1)
        idx.set_centroids(xb[:nlist])
        idx.add(len(xb), xb)
        prm = hx.make_params(nprobe=4, algo=hx.ALGO_BATCHED)
        q = torch.from_numpy(xq).cuda()
        D = torch.empty(n, k, device="cuda")
        I = torch.empty(n, k, dtype=torch.int64, device="cuda")
        torch.cuda.synchronize()
        idx.search_device(n, q.data_ptr(), k, D.data_ptr(), I.data_ptr(), prm, stats=True)
        # past the pinned size: the stages of host calls at their largest too
        idx.search(n, xq, 1000, params=prm)
        took = []
        for _ in range(3):
            t = time.perf_counter()
            for m in range(1, n, 7):
                Dm, Im, _ = idx.search(m, xq[:m], k, params=prm)
            took.append(time.perf_counter() - t)
        assert np.array_equal(Im, I.cpu().numpy()[:m]) and np.array_equal(Dm, D.cpu().numpy()[:m])
        ratios.append(took[0] / min(took[1:]))
    print(f"[time] first pass / later {ratios}", flush=True)
    assert min(ratios) < 1.4
