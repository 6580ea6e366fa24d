"""The selection by a workgroup per query at the edges of its forms, against
the oracle: survivor counts around the wave form's 1024, the registers' 2048
and several spans of them, k around the largest it sorts (256), tied distances,
exact (integer) and approximate (real, split scan) keys, batches just below
and above the size that a wave per query serves first.  Ids and distances bit
for bit."""
import numpy as np
import pytest

import oracle
from harmonyclient_amd import index as hx

pytestmark = pytest.mark.gpu


def _check(rows, d, n, k, data, metric=1, algo=hx.ALGO_BATCHED, nlist=1, P=1, tau=hx.TAU_NONE):
    print(f"[case] {data} {rows} x {d} nlist={nlist} n={n} k={k} metric={metric} algo={algo}", flush=True)
    r = np.random.default_rng(rows + k + n)
    xb, xq = (r.normal(0, 40, (m, d)) + 100 for m in (rows, n))
    if data == "int":
        xb, xq = (np.clip(np.rint(x), 0, 255) for x in (xb, xq))
    elif data == "dup":
        xb = np.clip(np.rint(xb[r.integers(0, 3, rows)]), 0, 255)
        xq = np.clip(np.rint(xq), 0, 255)
    xb, xq = xb.astype(np.float32), xq.astype(np.float32)
    cent = xb[r.permutation(rows)[:nlist]].copy()
    ix = oracle.Index.build(metric, xb, cent)
    idx = hx.Index(d, nlist, P, metric)
    idx.set_centroids(cent)
    idx.add(rows, xb)
    m = min(n, 64)
    OD, OI, _ = ix.search(xq[:m], P, k)
    D, I, st = idx.search(n, xq, k, params=hx.make_params(nprobe=P, algo=algo, tau=tau))
    assert np.array_equal(I[:m], OI), f"{(I[:m] != OI).sum()} ids differ"
    assert np.array_equal(D[:m].view(np.uint32), OD.view(np.uint32))
    if n > m:  # the same queries in a small batch
        t = slice(n - m, n)
        D2, I2, _ = idx.search(m, xq[t], k, params=hx.make_params(nprobe=P, algo=algo, tau=tau))
        assert np.array_equal(I[t], I2) and np.array_equal(D[t], D2)


@pytest.mark.parametrize("data", ["int", "real", "dup"])
@pytest.mark.parametrize("rows", [40, 1024, 1025, 2047, 2048, 2049, 4097, 9000])
@pytest.mark.parametrize("k", [1, 100, 256, 257])
def test_survivors(rows, data, k):
    _check(rows, 20, 5, k, data)


@pytest.mark.parametrize("n", [3071, 3072, 3073])
@pytest.mark.parametrize("data,rows", [("int", 900), ("real", 900), ("real", 1100), ("dup", 1100)])
def test_batch_sizes(n, data, rows):
    _check(rows, 12, n, 30, data)


@pytest.mark.parametrize("metric", [0, 1])
@pytest.mark.parametrize("n", [600, 3100])
def test_split_keys(metric, n):
    _check(24000, 72, n, 40, "real", metric, hx.ALGO_PLAIN, 16, 6, hx.TAU_WARMUP)
