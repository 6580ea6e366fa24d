"""List-major FP32 scan with overflowing inner products: a work item's slots
past its queries hold no query, so the rows that query 0 would rank below every
finite value (an inner product of +inf) must reach its results once each, and
only from the lists it probes.  Query counts per list that are no multiple of
the group size, fewer probes than lists; against the oracle and against each
query searched alone (a workgroup per list, without slots)."""
import numpy as np
import pytest

import oracle
from harmonyclient_amd import index as hx

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows,d,nlist,n,P,k,scale", [
    (6000, 516, 16, 1003, 8, 30, 1.0),   # past 512 dims
    (9000, 24, 16, 1003, 8, 300, 4e18),  # row norms past the split scan's range
])
def test_overflowing_products_and_absent_slots(rows, d, nlist, n, P, k, scale):
    print(f"[case] rows={rows} d={d} nlist={nlist} n={n} P={P} k={k} scale={scale}", flush=True)
    r = np.random.default_rng(d)
    c = r.normal(0, 1, (nlist, d))
    xb = ((c[r.integers(0, nlist, rows)] + 0.3 * r.normal(0, 1, (rows, d)) + 2.0) * scale).astype(np.float32)
    xq = (c[r.integers(0, nlist, n)] + 0.3 * r.normal(0, 1, (n, d))).astype(np.float32)
    xq[0] = np.float32(3e38 / scale) * np.sign(c[3] + 2.0)  # most rows' product overflows
    xq[17] = xq[0]
    xq[17, ::2] = 0.0
    ix = oracle.Index.build(0, xb, xb[:nlist].copy())
    idx = hx.Index(d, nlist, P, 0)
    idx.set_centroids(xb[:nlist])
    idx.add(rows, xb)
    OD, OI, _ = ix.search(xq, P, k)
    assert np.isposinf(OD[0]).sum() >= k // 2
    D, I, _ = idx.search(n, xq, k, params=hx.make_params(nprobe=P))
    for q in (0, 17):  # alone first: the batch's own faults are then told apart
        D1, I1, _ = idx.search(1, xq[q:q + 1], k, params=hx.make_params(nprobe=P))
        assert np.array_equal(I1[0], OI[q]) and np.array_equal(D1[0].view(np.uint32), OD[q].view(np.uint32)), f"query {q} alone"
    assert np.array_equal(I, OI), f"{(I != OI).sum()} ids differ, in queries {np.unique(np.nonzero(I != OI)[0])[:8]}"
    assert np.array_equal(D.view(np.uint32), OD.view(np.uint32))
