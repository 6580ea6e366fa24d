"""Plain and pruned searches of a batch (the exact FP32 scans and the split
MFMA scan, with their bound, plan and selection) against the oracle, over the forms those searches accept:
both metrics, odd dimensions, a query alone and queries that share lists,
per-query probe counts, k past the candidates, rows with many equal distances
(more survivors than a query's buffer holds), empty lists.  Ids and distances
bit for bit."""
import numpy as np
import pytest

import oracle
from harmonyclient_amd import index as hx

pytestmark = pytest.mark.gpu


def _data(kind, n, d, ncomp, seed):
    r = np.random.default_rng(seed)
    if kind == "dup":
        return np.rint(r.uniform(0, 3, (4, d)))[r.integers(0, 4, n)].astype(np.float32)
    c = r.uniform(0, 255, (ncomp, d))
    x = c[r.integers(0, ncomp, n)] + r.normal(0, 20, (n, d))
    if kind == "int":
        return np.clip(np.rint(x), 0, 255).astype(np.float32)
    if kind == "unit":
        x = x - 127.5
        return (x / np.linalg.norm(x, axis=1, keepdims=True)).astype(np.float32)
    return (x - 100.0).astype(np.float32)


def _index(kind, rows, d, nlist, metric, seed=1):
    xb = _data(kind, rows, d, max(nlist // 2, 1), seed)
    cent = xb[np.random.default_rng(seed).permutation(rows)[:nlist]].copy()
    if nlist > 3:
        cent[3] = 9e3  # a list without rows
    ix = oracle.Index.build(metric, xb, cent)
    idx = hx.Index(d, nlist, 1, metric)
    idx.set_centroids(cent)
    idx.add(rows, xb)
    return idx, ix


def _same(D, I, OD, OI):
    assert np.array_equal(I, OI), f"{(I != OI).sum()} ids differ"
    assert np.array_equal(D.view(np.uint32), OD.view(np.uint32))


@pytest.mark.parametrize("kind,rows,d,nlist,metric,n,P,k", [
    ("int", 4000, 128, 20, 1, 1, 8, 10), ("int", 4000, 128, 20, 1, 700, 20, 100), ("real", 6000, 17, 30, 1, 900, 12, 33),
    ("real", 5000, 3, 16, 1, 40, 16, 5), ("real", 3000, 1, 12, 1, 1200, 12, 7), ("unit", 5000, 130, 20, 0, 900, 9, 50),
    ("unit", 2000, 201, 25, 0, 6, 25, 300), ("int", 3000, 96, 10, 0, 1500, 10, 1), ("real", 2500, 420, 16, 1, 1500, 16, 64),
    ("real", 900, 600, 8, 1, 1500, 8, 20), ("real", 900, 600, 8, 0, 3, 8, 20), ("int", 700, 32, 30, 1, 2500, 30, 1000),
    ("int", 600, 32, 30, 0, 2, 30, 1024), ("dup", 24000, 16, 6, 1, 300, 6, 20), ("dup", 24000, 16, 6, 0, 2, 6, 20),
    ("int", 70, 8, 5, 1, 33, 1, 3), ("real", 40000, 64, 4, 1, 65, 4, 400),
])
def test_plain_batches(kind, rows, d, nlist, metric, n, P, k):
    print(f"[case] plain {kind} rows={rows} d={d} nlist={nlist} metric={metric} n={n} P={P} k={k}", flush=True)
    idx, ix = _index(kind, rows, d, nlist, metric)
    xq = _data(kind, n, d, max(nlist // 2, 1), 77)
    OD, OI, ost = ix.search(xq, P, k)
    D, I, st = idx.search(n, xq, k, params=hx.make_params(nprobe=P))
    _same(D, I, OD, OI)
    assert st.candidates == ost.candidates and st.blocks_total == st.candidates and st.blocks_skipped == 0
    if metric == 1:
        for tau in (hx.TAU_WARMUP, hx.TAU_NONE):
            for blk in (0, 5):
                prm = hx.make_params(nprobe=P, algo=hx.ALGO_PRUNED, tau=tau, dim_block=blk, warmup_lists=2)
                D, I, st = idx.search(n, xq, k, params=prm)
                _same(D, I, OD, OI)
                nb = -(-d // min(blk, d)) if blk else (4 if d >= 4 else 1)
                assert st.candidates == ost.candidates and st.blocks_total == nb * st.candidates
                assert 0 <= st.blocks_skipped <= (nb - 1) * st.candidates


@pytest.mark.parametrize("kind,rows,d,nlist,metric,n,P,k", [
    # sizes of the split scan: a wave's 64 and 128 dims, its last whole and
    # partial chunks, the workgroup form with odd and even chunk groups
    ("int", 30000, 64, 16, 1, 2500, 12, 20), ("real", 30000, 65, 16, 1, 2500, 12, 20), ("real", 30000, 113, 16, 1, 1300, 16, 130),
    ("unit", 30000, 128, 16, 0, 1300, 16, 50), ("int", 30000, 129, 16, 1, 1300, 16, 10), ("real", 16000, 240, 12, 1, 1600, 12, 256),
    ("unit", 12000, 300, 12, 0, 2000, 12, 30), ("real", 9000, 512, 12, 1, 1900, 12, 100), ("int", 20000, 250, 9, 0, 1500, 9, 7),
    ("dup", 33000, 130, 7, 1, 1100, 7, 12), ("dup", 33000, 40, 7, 0, 4100, 7, 300), ("int", 150, 128, 3, 1, 60000, 3, 4),
])
def test_split_batches_device(kind, rows, d, nlist, metric, n, P, k):
    """The device entry point without statistics (plain, and pruned for L2)."""
    import torch
    print(f"[case] split {kind} rows={rows} d={d} nlist={nlist} metric={metric} n={n} P={P} k={k}", flush=True)
    idx, ix = _index(kind, rows, d, nlist, metric)
    xq = _data(kind, n, d, max(nlist // 2, 1), 78)
    OD, OI, _ = ix.search(xq, P, k)
    q = torch.from_numpy(xq).cuda()
    for algo in (hx.ALGO_PLAIN, hx.ALGO_PRUNED)[:1 + metric]:
        D = torch.full((n, k), -7.0, device="cuda")
        I = torch.full((n, k), -7, dtype=torch.int64, device="cuda")
        torch.cuda.synchronize()
        idx.search_device(n, q.data_ptr(), k, D.data_ptr(), I.data_ptr(), hx.make_params(nprobe=P, algo=algo), stats=False)
        torch.cuda.synchronize()
        _same(D.cpu().numpy(), I.cpu().numpy(), OD, OI)


def test_split_margin_and_non_finite_queries():
    """Rows whose distances differ by less than the split ranks resolve (large
    common offset), queries with inf, NaN and overflowing norms among them."""
    import torch
    print("[case] split: offset 4096 +- 1e-2, non-finite queries", flush=True)
    r = np.random.default_rng(5)
    rows, d, n, P, k = 30000, 100, 2000, 12, 40
    xb = (4096.0 + 1e-2 * r.normal(0, 1, (rows, d))).astype(np.float32)
    cent = xb[:16].copy()
    ix = oracle.Index.build(1, xb, cent)
    idx = hx.Index(d, 16, 1)
    idx.set_centroids(cent)
    idx.add(rows, xb)
    xq = (4096.0 + 1e-2 * r.normal(0, 1, (n, d))).astype(np.float32)
    xq[3, 5], xq[70, 0], xq[71] = np.nan, np.inf, 1e19
    OD, OI, _ = ix.search(xq, P, k)
    q = torch.from_numpy(xq).cuda()
    D = torch.empty(n, k, device="cuda")
    I = torch.empty(n, k, dtype=torch.int64, device="cuda")
    torch.cuda.synchronize()
    idx.search_device(n, q.data_ptr(), k, D.data_ptr(), I.data_ptr(), hx.make_params(nprobe=P), stats=False)
    torch.cuda.synchronize()
    _same(D.cpu().numpy(), I.cpu().numpy(), OD, OI)


@pytest.mark.parametrize("metric", [1, 0])
def test_per_query_probe_counts_and_replay(metric):
    """Per-query probe counts (0 and past nprobe among them) read on the
    device, and replays of the captured search with new queries."""
    import torch
    print(f"[case] plain per-query nprobe, captured, metric={metric}", flush=True)
    idx, ix = _index("int", 8000, 48, 24, metric)
    n, P, k = 800, 16, 40
    npq = np.random.default_rng(3).integers(0, P + 3, n).astype(np.int32)
    st = torch.cuda.Stream()
    with torch.cuda.stream(st):
        q = torch.empty(n, 48, device="cuda")
        c = torch.from_numpy(npq).cuda()
        D = torch.empty(n, k, device="cuda")
        I = torch.empty(n, k, dtype=torch.int64, device="cuda")
        prm = hx.make_params(nprobe=P, use_graph=True, nprobe_per_query_dev=c.data_ptr())
        for rep in range(4):
            xq = _data("int", n, 48, 12, 50 + rep)
            q.copy_(torch.from_numpy(xq))
            idx.search_device(n, q.data_ptr(), k, D.data_ptr(), I.data_ptr(), prm, stats=False, stream=st.cuda_stream)
            st.synchronize()
            OD = np.full((n, k), np.finfo(np.float32).max if metric else -np.finfo(np.float32).max, np.float32)
            OI = np.full((n, k), -1, np.int64)
            for p in np.unique(np.clip(npq, 0, P)):
                rows = np.flatnonzero(np.clip(npq, 0, P) == p)
                if p > 0:
                    OD[rows], OI[rows], _ = ix.search(np.ascontiguousarray(xq[rows]), int(p), k)
            _same(D.cpu().numpy(), I.cpu().numpy(), OD, OI)
            if rep == 1:  # another search of the handle between the replays
                idx.search(20, xq[:20], 5, params=hx.make_params(nprobe=3))


def test_infinite_and_nan_values():
    """Rows and queries with inf, NaN and values whose distances overflow: as
    the oracle's strict admission (never inf or NaN)."""
    print("[case] plain: inf / NaN / overflowing rows and queries", flush=True)
    idx, _ = _index("real", 3000, 20, 16, 1, 2)
    off, ids, codes = idx.csr()
    codes = codes.copy()
    codes[::11, 4] = np.inf
    codes[5::17, 2] = np.nan
    codes[7::13] *= np.float32(1e19)
    idx.set_lists(off, ids, codes)
    ix = oracle.Index(1, idx.centroids, off, ids, codes)
    for n in (2, 1500):
        xq = _data("real", n, 20, 8, 60)
        xq[0, 1] = np.inf
        xq[1] = codes[7] if n == 2 else xq[1]
        xq[n // 2:n // 2 + 1, 3] = np.nan
        OD, OI, _ = ix.search(xq, 16, 30)
        D, I, _ = idx.search(n, xq, 30, params=hx.make_params(nprobe=16))
        _same(D, I, OD, OI)
