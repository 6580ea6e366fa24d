"""GPU index build against the oracle: row assignment (the MFMA form with its
exact rescoring and its hand-over to the per-query kernel), list order and
k-means.  Labels, order, ids and distances are exact on both sides, so every
comparison is bit for bit."""
import numpy as np
import pytest

import oracle
from harmonyclient_amd import index as hx

pytestmark = pytest.mark.gpu


def _rows(kind, n, d, nlist, seed):
    r = np.random.default_rng(seed)
    if kind == "int":
        c = np.rint(r.uniform(0, 255, (max(nlist // 2, 1), d)))
        x = np.clip(np.rint(c[r.integers(0, len(c), n)] + r.normal(0, 20, (n, d))), 0, 255)
    elif kind == "dup":  # a handful of distinct rows: exact ties between centroids everywhere
        x = np.rint(r.uniform(0, 4, (7, d)))[r.integers(0, 7, n)]
    elif kind == "near":  # centroids that differ by less than the approximation resolves
        x = 100.0 + 1e-4 * r.normal(0, 1, (n, d))
    else:
        x = r.standard_t(3, (n, d)) * np.exp(r.normal(0, 1, d))
    return np.ascontiguousarray(x, np.float32)


@pytest.mark.parametrize("metric", [hx.METRIC_L2, hx.METRIC_IP])
@pytest.mark.parametrize("kind,n,d,nlist", [
    ("int", 5000, 128, 100), ("int", 257, 1, 33), ("real", 255, 17, 1), ("real", 4097, 128, 65),
    ("real", 1000, 129, 40), ("real", 1000, 200, 32), ("dup", 1500, 24, 31), ("near", 700, 64, 50),
    ("real", 600, 420, 97), ("int", 1, 96, 5), ("real", 300, 512, 20), ("real", 200, 516, 20),
    ("int", 250_000, 17, 24),  # an upload in pinned chunks, rows padded on the way
])
def test_add_assignment(metric, kind, n, d, nlist):
    print(f"[case] add {kind} n={n} d={d} nlist={nlist} metric={metric}", flush=True)
    x = _rows(kind, n, d, nlist, 5 + d)
    cent = x[np.random.default_rng(9).permutation(n)[:nlist]] if n >= nlist else _rows(kind, nlist, d, nlist, 3)
    idx = hx.Index(d, nlist, 1, metric)
    idx.set_centroids(cent)
    idx.add(n, x)
    off, ids, codes = idx.csr()
    ix = oracle.Index.build(metric, x, cent)
    assert np.array_equal(off, ix.list_off)
    assert np.array_equal(ids, ix.ids)
    assert np.array_equal(codes, ix.codes)


@pytest.mark.parametrize("metric", [hx.METRIC_L2, hx.METRIC_IP])
@pytest.mark.parametrize("kind,n,d,nlist", [("int", 3000, 30, 40), ("real", 2049, 128, 64), ("dup", 900, 20, 16)])
def test_train_rounds(metric, kind, n, d, nlist):
    print(f"[case] train {kind} n={n} d={d} nlist={nlist} metric={metric}", flush=True)
    x = _rows(kind, n, d, nlist, 11)
    init = x[np.random.default_rng(2).permutation(n)[:nlist]]
    idx = hx.Index(d, nlist, 1, metric)
    idx.train(n, x, init_centroids=init, niter=4)
    assert np.array_equal(idx.centroids.view(np.uint32), oracle.kmeans(metric, x, init, 4).view(np.uint32))


@pytest.mark.parametrize("scale", [1e18, 1e16, np.nan])
def test_assignment_of_large_and_non_finite_rows(scale):
    """Norms beyond the approximation's range go through the exact kernel; a
    row with no finite distance to any centroid (the oracle's chain overflows
    for some of the 1e18 rows) is refused, as by the exact kernel alone."""
    print(f"[case] add: rows scaled by {scale}", flush=True)
    x = _rows("real", 300, 32, 10, 4)
    x[::7] *= np.float32(scale)
    cent = x[:10].copy() if np.isfinite(scale) else _rows("real", 10, 32, 10, 6)
    idx = hx.Index(32, 10, 1)
    idx.set_centroids(cent)
    _, labels = oracle.coarse(oracle.METRIC_L2, x, cent, 1)
    if (labels < 0).any():
        with pytest.raises(hx.HivfError):
            idx.add(300, x)
        return
    assert scale == 1e16
    ix = oracle.Index.build(oracle.METRIC_L2, x, cent)
    idx.add(300, x)
    off, ids, _ = idx.csr()
    assert np.array_equal(off, ix.list_off) and np.array_equal(ids, ix.ids)
