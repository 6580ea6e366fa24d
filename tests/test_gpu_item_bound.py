"""The work-item tables of batched and list-major searches: sized by what the
probes can reach (one long list among many short ones takes no table as if all
were long), and large enough where every query probes the longest lists, at
query counts around an item's.  Ids and distances against the oracle."""
import numpy as np
import pytest

import oracle
from harmonyclient_amd import index as hx

pytestmark = pytest.mark.gpu


def _skewed(long_rows, short_rows, nlist, d, seed, real=False):
    r = np.random.default_rng(seed)
    cent = r.uniform(0, 255, (nlist, d))
    cent[0] = 128.0
    x = np.concatenate([cent[0] + r.normal(0, 6, (long_rows, d)),
                        cent[r.integers(1, nlist, short_rows)] + r.normal(0, 2, (short_rows, d))])
    if not real:
        x, cent = np.clip(np.rint(x), 0, 255), np.rint(cent)
    return x.astype(np.float32), cent.astype(np.float32), r


def _build(xb, cent):
    idx = hx.Index(cent.shape[1], cent.shape[0], 1, 1)
    idx.set_centroids(cent)
    idx.add(xb.shape[0], xb)
    return idx


@pytest.mark.parametrize("algo,limit_mb", [(hx.ALGO_BATCHED, 140), (hx.ALGO_PLAIN, 620)])
def test_one_long_list_takes_no_table_as_if_all_were(algo, limit_mb):
    """(With a batched search's shadows, 75 MB here, and a plain search's survivor
    buffers, 131 KB for each of 4000 queries.)"""
    import torch
    print(f"[case] table of one list of 400k rows among 4096, algo={algo}", flush=True)
    xb, cent, r = _skewed(400_000, 40_000, 4096, 8, 1)
    n, P, k = 4000, 32, 10
    idx = _build(xb, cent)
    xq = xb[r.integers(0, len(xb), n)]
    prm = hx.make_params(nprobe=P, algo=algo, survivor_cap=64 if algo == hx.ALGO_BATCHED else 0)
    idx.coarse(xq, P)
    torch.cuda.synchronize()
    free = torch.cuda.mem_get_info()[0]
    D, I, _ = idx.search(n, xq, k, params=prm)
    used = (free - torch.cuda.mem_get_info()[0]) / 1e6
    print(f"[memory] {used:.0f} MB", flush=True)
    OD, OI, _ = oracle.Index.build(1, xb, cent).search(xq[:20], P, k)
    assert np.array_equal(I[:20], OI) and np.array_equal(D[:20], OD)
    assert used < limit_mb


@pytest.mark.parametrize("n", [31, 32, 33, 64, 65, 1000, 3200])
@pytest.mark.parametrize("P,rows", [(1, 30_000), (3, 9_000), (24, 3_000)])
@pytest.mark.parametrize("real", [False, True])
def test_every_query_probes_the_longest_lists(n, P, rows, real):
    print(f"[case] n={n} P={P} rows={rows} real={real}", flush=True)
    xb, cent, r = _skewed(rows, 600, 24, 12, n + P, real)
    idx = _build(xb, cent)
    xq = (128.0 + r.normal(0, 3, (n, 12))).astype(np.float32)
    if not real:
        xq = np.rint(xq)
    k = 20
    m = min(n, 40)
    OD, OI, _ = oracle.Index.build(1, xb, cent).search(xq[-m:], P, k)
    for kw in (dict(algo=hx.ALGO_BATCHED), dict(algo=hx.ALGO_BATCHED, batch_queries=32, batch_rows=32),
               dict(algo=hx.ALGO_BATCHED, batch_queries=64, batch_rows=96, precision=hx.PREC_BF16), dict(algo=hx.ALGO_PLAIN)):
        D, I, _ = idx.search(n, xq, k, params=hx.make_params(nprobe=P, **kw))
        assert np.array_equal(I[-m:], OI) and np.array_equal(D[-m:].view(np.uint32), OD.view(np.uint32)), kw
