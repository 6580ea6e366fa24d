"""Batched searches of real-valued lists (the FP16 shadow, its error bound and
the selection of its approximate keys) against the oracle: magnitudes at both
ends of the shadow's range and past it, values far below a list's largest,
a common offset that leaves the bound wide, queries that FP16 cannot hold, odd
dimensions, one query, more survivors than a wave holds in registers, k past
the wave form's limit.  Ids and distances bit for bit."""
import numpy as np
import pytest

import oracle
from harmonyclient_amd import index as hx

pytestmark = pytest.mark.gpu


def _data(rows, d, ncomp, scale, offset, spread, seed):
    r = np.random.default_rng(seed)
    c = r.normal(0, 3, (ncomp, d))
    x = c[r.integers(0, ncomp, rows)] + r.standard_t(3.0, (rows, d))
    x *= np.exp2(-r.integers(0, spread + 1, d))  # dimensions of smaller magnitude
    return (x * scale + offset).astype(np.float32)


@pytest.mark.parametrize("rows,d,nlist,n,P,k,scale,offset,spread", [
    (3000, 16, 12, 70, 12, 10, 1.0, 0.0, 0), (3000, 17, 12, 33, 5, 3, 1.0, 0.0, 0), (2500, 128, 10, 1, 10, 20, 1.0, 0.0, 0),
    (2500, 129, 10, 300, 1, 20, 1.0, 0.0, 0), (1500, 256, 9, 65, 9, 64, 1.0, 0.0, 0), (1500, 257, 9, 64, 9, 64, 1.0, 0.0, 0),
    (1200, 512, 8, 40, 8, 30, 1.0, 0.0, 0), (900, 1, 8, 40, 8, 5, 1.0, 0.0, 0), (4000, 24, 10, 50, 10, 256, 1.0, 0.0, 0),
    (4000, 24, 10, 50, 10, 300, 1.0, 0.0, 0), (3000, 32, 10, 60, 10, 10, 1e-9, 0.0, 0), (3000, 32, 10, 60, 10, 10, 1e-16, 0.0, 0),
    (3000, 32, 10, 60, 10, 10, 1e12, 0.0, 0), (3000, 32, 10, 60, 10, 10, 1e14, 0.0, 0), (3000, 48, 10, 60, 10, 10, 1.0, 0.0, 30),
    (6000, 64, 4, 60, 4, 10, 1.0, 500.0, 0), (30000, 20, 4, 40, 4, 10, 1.0, 3000.0, 0),
])
def test_batched_real(rows, d, nlist, n, P, k, scale, offset, spread):
    print(f"[case] {rows} x {d} nlist={nlist} n={n} P={P} k={k} scale={scale} offset={offset} spread={spread}", flush=True)
    xb = _data(rows, d, nlist, scale, offset, spread, 5)
    cent = xb[np.random.default_rng(1).permutation(rows)[:nlist]].copy()
    xq = _data(n, d, nlist, scale, offset, spread, 6)
    if n > 4:
        xq[1] *= np.float32(1e4)  # past FP16 at the lists' scale
        xq[2] = 0.0
        xq[3] *= np.float32(1e-4)
    ix = oracle.Index.build(1, xb, cent)
    idx = hx.Index(d, nlist, 1, 1)
    idx.set_centroids(cent)
    idx.add(rows, xb)
    OD, OI, _ = ix.search(xq, P, k)
    for tau in (hx.TAU_WARMUP, hx.TAU_NONE):  # TAU_NONE: every probed row survives
        for rpi in (0, 64):
            D, I, _ = idx.search(n, xq, k, params=hx.make_params(nprobe=P, algo=hx.ALGO_BATCHED, tau=tau, batch_rows=rpi))
            assert np.array_equal(I, OI), f"{(I != OI).sum()} ids differ"
            assert np.array_equal(D.view(np.uint32), OD.view(np.uint32))


@pytest.mark.parametrize("data", ["int", "mixed", "real", "dup"])
@pytest.mark.parametrize("d", [3, 128, 200, 420])
@pytest.mark.parametrize("L,W,k", [(0, 0, 1), (0, 0, 50), (3, 33, 100), (1, 64, 65), (5, 1000, 200), (12, 340, 400), (40, 70, 30)])
def test_warmup_from_the_shadow(d, data, L, W, k):
    """The bound from the shadow's first rows: lists shorter and longer than
    the rows taken, counts around whole tiles, fewer rows than k (no bound),
    more than the kernel holds (the FP32 scan's bound), queries that are not
    integer among integer ones."""
    print(f"[case] warm {data} d={d} L={L} W={W} k={k}", flush=True)
    rows, nlist, n, P = 5000, 20, 70, 12
    r = np.random.default_rng(d + k)
    xb, xq = (r.normal(0, 40, (m, d)) + 100 for m in (rows, n))
    if data != "real":
        xb, xq = (np.clip(np.rint(x), 0, 255) for x in (xb, xq))
    if data == "mixed":
        xq[::5] += 0.25
    if data == "dup":
        xb = xb[r.integers(0, 30, rows)]
    xb, xq = xb.astype(np.float32), xq.astype(np.float32)
    cent = xb[r.permutation(rows)[:nlist]].copy() if data != "dup" else np.clip(np.rint(r.normal(0, 40, (nlist, d)) + 100), 0, 255).astype(np.float32)
    ix = oracle.Index.build(1, xb, cent)
    idx = hx.Index(d, nlist, 1, 1)
    idx.set_centroids(cent)
    idx.add(rows, xb)
    OD, OI, _ = ix.search(xq, P, k)
    D, I, st = idx.search(n, xq, k, params=hx.make_params(nprobe=P, algo=hx.ALGO_BATCHED, tau=hx.TAU_WARMUP, warmup_lists=L,
                                                          warmup_list_size=W))
    assert np.array_equal(I, OI), f"{(I != OI).sum()} ids differ"
    assert np.array_equal(D.view(np.uint32), OD.view(np.uint32))
    assert st.exact_rescans == 0
