"""Host searches around the size that pinned buffers serve (2 MiB of queries
and results), growing and shrinking from call to call, against the device
search of the same queries; counters as many as with device buffers."""
import numpy as np
import pytest
import torch

from harmonyclient_amd import index as hx

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("algo,metric", [(hx.ALGO_PLAIN, 0), (hx.ALGO_PRUNED, 1), (hx.ALGO_BATCHED, 1)])
@pytest.mark.parametrize("d", [30, 64])
def test_sizes(algo, metric, d):
    rows, nlist, P, k = 3000, 16, 5, 40
    r = np.random.default_rng(d)
    xb = r.normal(0, 30, (rows, d)).astype(np.float32)
    idx = hx.Index(d, nlist, P, metric)
    idx.set_centroids(xb[:nlist].copy())
    idx.add(rows, xb)
    edge = (2 << 20) // (4 * d + 12 * k)
    prm = hx.make_params(nprobe=P, algo=algo)
    for n in (1, edge - 1, 3, edge, edge + 1, 7, 2 * edge, 1):
        print(f"[case] n={n} d={d} algo={algo}", flush=True)
        xq = r.normal(0, 30, (n, d)).astype(np.float32)
        D, I, st = idx.search(n, xq, k, params=prm)
        q = torch.from_numpy(xq).cuda()
        oD, oI = torch.empty(n, k, device="cuda"), torch.empty(n, k, dtype=torch.int64, device="cuda")
        st2 = idx.search_device(n, q.data_ptr(), k, oD.data_ptr(), oI.data_ptr(), prm, stats=True)
        torch.cuda.synchronize()
        assert np.array_equal(D.view(np.uint32), oD.cpu().numpy().view(np.uint32)) and np.array_equal(I, oI.cpu().numpy())
        assert (st.candidates, st.survivors, st.scan_kind) == (st2.candidates, st2.survivors, st2.scan_kind)
