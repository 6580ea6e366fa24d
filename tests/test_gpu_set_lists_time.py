"""Lists set verbatim: their largest value, integer check and norms are found in
about the time numpy takes on one thread, however many lists share the threads;
and the forms chosen from them are those of the same rows added (inf and NaN, a
value past the norms' range and real values in one list each)."""
import time

import numpy as np
import pytest

import oracle
from harmonyclient_amd import index as hx

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows,d,nlist", [(500_000, 3, 50), (60_000, 128, 64)])
def test_time_of_set_lists(rows, d, nlist):
    print(f"[case] set_lists {rows} x {d} nlist={nlist}", flush=True)
    codes = np.random.default_rng(1).normal(0, 1, (rows, d)).astype(np.float32)
    off = np.linspace(0, rows, nlist + 1).astype(np.int64)
    ids = np.arange(rows)
    idx = hx.Index(d, nlist, 1, 1)
    idx.set_centroids(codes[:nlist])

    def best(f):
        t = []
        for _ in range(5):
            t0 = time.perf_counter()
            f()
            t.append(time.perf_counter() - t0)
        return min(t)

    def alone():
        (codes.astype(np.float64) ** 2).sum(1).astype(np.float32)
        np.abs(codes).max()
        ((codes >= 0) & (codes <= 255) & (codes == np.rint(codes))).all()
        codes.copy()

    a, b = best(lambda: idx.set_lists(off, ids, codes)), best(alone)
    print(f"[time] set_lists {a * 1e3:.1f} ms, numpy {b * 1e3:.1f} ms", flush=True)
    assert a < b


@pytest.mark.parametrize("value", [None, 0.5, 1e19, np.inf, np.nan, -1.0, 256.0])
def test_forms_of_set_lists(value):
    print(f"[case] one value {value} in integer lists", flush=True)
    r = np.random.default_rng(2)
    rows, d, nlist, n, P, k = 3000, 24, 12, 400, 12, 10
    xb = np.rint(r.uniform(0, 255, (rows, d))).astype(np.float32)
    xq = np.rint(r.uniform(0, 255, (n, d))).astype(np.float32)
    idx = hx.Index(d, nlist, 1, 1)
    idx.set_centroids(xb[:nlist])
    idx.add(rows, xb)
    off, ids, codes = idx.csr()
    codes = codes.copy()
    if value is not None:
        codes[1700, 7] = value
    idx.set_lists(off, ids, codes)
    ix = oracle.Index(1, xb[:nlist], off, ids, codes)
    OD, OI, _ = ix.search(xq, P, k)
    for algo in (hx.ALGO_PLAIN, hx.ALGO_BATCHED):
        D, I, st = idx.search(n, xq, k, params=hx.make_params(nprobe=P, algo=algo))
        assert np.array_equal(I, OI) and np.array_equal(D.view(np.uint32), OD.view(np.uint32))
    assert (st.scan_kind == 2) == (value is None)
