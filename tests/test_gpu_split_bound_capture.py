"""Lists set anew and searched for the first time under a caller's stream capture:
nothing waits for the lists' error bound there, the replays give the exact results,
and the first search outside asks for it."""
import numpy as np
import pytest

from harmonyclient_amd import index as hx

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("algo", [hx.ALGO_PLAIN, hx.ALGO_PRUNED])
def test_first_search_of_new_lists_captured(algo):
    print(f"[case] algo={algo}", flush=True)
    d, nlist, rows, n, P, k = 64, 64, 700, 1000, 16, 20
    r = np.random.default_rng(5)
    c = r.normal(0, 3, (nlist, d)).astype(np.float32)
    off, ids = np.arange(nlist + 1) * rows, np.arange(nlist * rows)

    def near(l):
        return (c[l] + r.normal(0, 1, (len(l), d))).astype(np.float32)

    idx = hx.Index(d, nlist, P, 1)
    idx.set_centroids(c)
    xq = near(r.integers(0, nlist, n))
    x = torch.from_numpy(xq).cuda()
    D = torch.empty(n, k, device="cuda")
    I = torch.empty(n, k, dtype=torch.int64, device="cuda")
    prm = hx.make_params(nprobe=P, algo=algo)
    s = torch.cuda.Stream()

    def run():
        idx.search_device(n, x.data_ptr(), k, D.data_ptr(), I.data_ptr(), prm, stats=False, stream=s.cuda_stream)

    for captured in (False, True):
        xb = near(np.repeat(np.arange(nlist), rows))
        idx.set_lists(off, ids, xb)
        _, pr = idx.coarse(xq, P)
        ED, EI, _ = idx.scan(xq, pr, k)
        torch.cuda.synchronize()
        if not captured:
            run()
        else:
            g = torch.cuda.CUDAGraph()
            with torch.cuda.graph(g, stream=s, capture_error_mode="thread_local"):
                run()
        for _ in range(3):
            D.zero_()
            I.zero_()
            torch.cuda.synchronize()
            if captured:
                g.replay()
            else:
                run()
            torch.cuda.synchronize()
            assert np.array_equal(I.cpu().numpy(), EI) and np.array_equal(D.cpu().numpy(), ED)
        run()
        torch.cuda.synchronize()
        assert np.array_equal(I.cpu().numpy(), EI) and np.array_equal(D.cpu().numpy(), ED)
