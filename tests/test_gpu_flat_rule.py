"""Plain and pruned batches on short lists, with statistics: the search must not
take a form that is much slower than a workgroup per query over its lists, which
the scan alone (the same probes and bounds) measures.  Results equal the scan's."""
import numpy as np
import pytest

from harmonyclient_amd import index as hx

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("d,rows,n,P,algo", [
    (32, 64, 1000, 32, hx.ALGO_PRUNED), (128, 16, 1000, 32, hx.ALGO_PRUNED), (300, 40, 1000, 32, hx.ALGO_PRUNED),
    (128, 200, 256, 16, hx.ALGO_PRUNED), (128, 16, 1000, 8, hx.ALGO_PLAIN), (300, 64, 256, 1, hx.ALGO_PLAIN),
    (128, 40, 1000, 2, hx.ALGO_PLAIN), (32, 128, 4000, 8, hx.ALGO_PLAIN), (128, 400, 1000, 32, hx.ALGO_PLAIN),
    (128, 400, 2000, 32, hx.ALGO_PRUNED),
])
def test_not_slower_than_a_workgroup_per_query(d, rows, n, P, algo):
    print(f"[case] d={d} rows={rows} n={n} P={P} algo={algo}", flush=True)
    nlist, k = 256, 10
    r = np.random.default_rng(d + rows)
    c = r.integers(0, 256, (nlist, d)).astype(np.float32)

    def near(l, s):
        return np.clip(np.rint(c[l] + r.normal(0, s, (len(l), d))), 0, 255).astype(np.float32)

    idx = hx.Index(d, nlist, P, 1)
    idx.set_centroids(c)
    idx.set_lists(np.arange(nlist + 1) * rows, np.arange(nlist * rows), near(np.repeat(np.arange(nlist), rows), 5))
    xq = near(r.integers(0, nlist, n), 20)
    _, pr = idx.coarse(xq, P)
    tau = idx.warmup_tau(xq, pr, k) if algo == hx.ALGO_PRUNED else None
    prm = hx.make_params(nprobe=P, algo=algo)
    search, alone = [], []
    for _ in range(9):
        D, I, st = idx.search(n, xq, k, params=prm)
        search.append(st.tau_ms + st.scan_ms)
        D1, I1, s1 = idx.scan(xq, pr, k, algo=algo, tau=tau)
        alone.append(s1.scan_ms)
    assert np.array_equal(I, I1) and np.array_equal(D, D1)
    print(f"[time] search {min(search) * 1e3:.0f} us, scan {min(alone) * 1e3:.0f} us", flush=True)
    # (the launches around the scan: a bound for the pruned form, events)
    assert min(search) < 1.4 * min(alone) + 0.03
