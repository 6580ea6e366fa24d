"""The form of plain and pruned batches on lists that the index built itself, whose
sizes differ and whose lists lie near one another: pruned searches take about the
plain search's time, and searches of large lists far less than a workgroup per query."""
import time

import numpy as np
import pytest

from harmonyclient_amd import index as hx

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


def _index(d, nlist, rows, clusters, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    c = torch.randn(clusters, d, device="cuda", generator=g) * (3.0 if clusters > 1 else 0.0)

    def data(n):
        return c[torch.randint(clusters, (n,), device="cuda", generator=g)] + torch.randn(n, d, device="cuda", generator=g)

    xb = data(rows).cpu().numpy()
    idx = hx.Index(d, nlist, 1, 1)
    idx.set_centroids(xb[:nlist])
    idx.add(rows, xb)
    return idx, data


def _time(idx, x, k, prm):
    n = x.shape[0]
    D = torch.empty(n, k, device="cuda")
    I = torch.empty(n, k, dtype=torch.int64, device="cuda")
    torch.cuda.synchronize()
    ms = []
    for _ in range(9):
        t0 = time.perf_counter()
        idx.search_device(n, x.data_ptr(), k, D.data_ptr(), I.data_ptr(), prm, stats=False)
        torch.cuda.synchronize()
        ms.append((time.perf_counter() - t0) * 1e3)
    return min(ms), D.cpu().numpy(), I.cpu().numpy()


@pytest.mark.parametrize("d,nlist,rows,clusters,n,P", [
    (96, 64, 300_000, 32, 600, 1), (128, 1000, 20_000, 500, 4000, 64), (201, 16, 20_000, 8, 20, 1),
])
def test_pruned_takes_about_the_plain_time(d, nlist, rows, clusters, n, P):
    print(f"[case] d={d} nlist={nlist} rows={rows} n={n} P={P}", flush=True)
    idx, data = _index(d, nlist, rows, clusters, d)
    x = data(n).contiguous()
    t = {a: _time(idx, x, 10, hx.make_params(nprobe=P, algo=a)) for a in (hx.ALGO_PLAIN, hx.ALGO_PRUNED)}
    p, q = t[hx.ALGO_PLAIN], t[hx.ALGO_PRUNED]
    assert np.array_equal(p[2], q[2]) and np.array_equal(p[1], q[1])
    print(f"[time] plain {p[0] * 1e3:.0f} us, pruned {q[0] * 1e3:.0f} us", flush=True)
    assert q[0] < 1.3 * p[0]


@pytest.mark.parametrize("algo", [hx.ALGO_PLAIN, hx.ALGO_PRUNED])
@pytest.mark.parametrize("d,nlist,rows,n,P", [(300, 256, 256_000, 4000, 1), (300, 256, 256_000, 600, 4), (300, 2000, 400_000, 4000, 4)])
def test_large_lists_are_shared(d, nlist, rows, n, P, algo):
    print(f"[case] d={d} nlist={nlist} n={n} P={P} algo={algo}", flush=True)
    idx, data = _index(d, nlist, rows, 1, 3)  # (Gaussian rows: the list of a row has several times the mean's)
    x = data(n).contiguous()
    t, D, I = _time(idx, x, 10, hx.make_params(nprobe=P, algo=algo))
    q = x.cpu().numpy()
    _, pr = idx.coarse(q, P)
    alone = []
    for _ in range(3):
        SD, SI, st = idx.scan(q, pr, 10)
        alone.append(st.scan_ms)
    assert np.array_equal(I, SI) and np.array_equal(D, SD)
    print(f"[time] search {t * 1e3:.0f} us, a workgroup per query {min(alone) * 1e3:.0f} us", flush=True)
    assert t < 0.5 * min(alone)
