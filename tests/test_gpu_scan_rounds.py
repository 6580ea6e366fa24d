"""The per-query scan at the sizes where its rounds change (k = 512 and 513) and
at its largest k, plain, pruned and warm-up, alone and as the rescan of queries
with more survivors than their buffer holds: against the oracle, and a large
k in little more time than a small one (the kept keys leave the buffer room)."""
import numpy as np
import pytest

import oracle
from harmonyclient_amd import index as hx

pytestmark = pytest.mark.gpu


def _index(rows, d, nlist, metric, seed):
    r = np.random.default_rng(seed)
    c = r.uniform(0, 255, (nlist, d))

    def data(m):
        return np.clip(np.rint(c[r.integers(0, nlist, m)] + r.normal(0, 20, (m, d))), 0, 255).astype(np.float32)

    xb = data(rows)
    cent = xb[:nlist].copy()
    idx = hx.Index(d, nlist, 1, metric)
    idx.set_centroids(cent)
    idx.add(rows, xb)
    return idx, oracle.Index.build(metric, xb, cent), data


@pytest.mark.parametrize("d", [3, 33, 64, 130])
@pytest.mark.parametrize("metric", [0, 1])
@pytest.mark.parametrize("k", [511, 512, 513, 1024])
def test_round_sizes(d, metric, k):
    print(f"[case] d={d} metric={metric} k={k}", flush=True)
    idx, ix, data = _index(9000, d, 20, metric, d + k)
    P = 12
    xq = data(9)
    OD, OI, _ = ix.search(xq, P, k)
    _, pr = idx.coarse(xq, P)
    for algo in (hx.ALGO_PLAIN, hx.ALGO_PRUNED)[:1 + metric]:
        D, I, _ = idx.scan(xq, pr, k, algo=algo)
        assert np.array_equal(I, OI) and np.array_equal(D.view(np.uint32), OD.view(np.uint32))
    for W in (1, 300, 2000):
        tau = idx.warmup_tau(xq, pr, k, L=P, W=W)
        assert np.array_equal(tau.view(np.uint32), ix.warmup_tau(xq, pr, k, P, W).view(np.uint32))
    if metric:
        for n in (3, 700):  # few listed queries: split; many: walked
            xq = data(n)
            OD, OI, _ = ix.search(xq[:30], P, k)
            prm = hx.make_params(nprobe=P, algo=hx.ALGO_BATCHED, survivor_cap=64)
            D, I, st = idx.search(n, xq, k, params=prm)
            assert st.exact_rescans > 0
            assert np.array_equal(I[:30], OI) and np.array_equal(D[:30].view(np.uint32), OD.view(np.uint32))


def test_large_k_keeps_its_rounds():
    print("[case] 64 queries of 32 lists, k = 100 and 1000", flush=True)
    idx, _, data = _index(500_000, 128, 1024, 1, 1)
    xq = data(64)
    _, pr = idx.coarse(xq, 32)
    ms = {k: min(idx.scan(xq, pr, k)[2].scan_ms for _ in range(9)) for k in (100, 1000)}
    print(f"[time] {ms}", flush=True)
    assert ms[1000] < 1.7 * ms[100]
