"""The selections at known survivor counts: with fewer warm-up rows than k there
is no bound and every probed row survives, so the counts are the list's rows,
around the wave form's 1024, the workgroup form's 2048 in registers and the
survivor buffer's size; batches served by a workgroup per query and by a wave.
Ids and distances against the oracle."""
import numpy as np
import pytest

import oracle
from harmonyclient_amd import index as hx

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("data", ["int", "bf16", "real", "dup"])
@pytest.mark.parametrize("rows", [60, 64, 1023, 1024, 1025, 2047, 2048, 2049, 4100])
@pytest.mark.parametrize("n,k", [(5, 2), (5, 256), (5, 257), (3100, 40), (3100, 256)])
def test_every_row_survives(rows, data, n, k):
    print(f"[case] {data} rows={rows} n={n} k={k}", flush=True)
    d = 20
    r = np.random.default_rng(rows + k)
    xb, xq = (r.normal(0, 40, (m, d)) + 100 for m in (rows, n))
    if data != "real":
        xb, xq = (np.clip(np.rint(x), 0, 255) for x in (xb, xq))
    if data == "dup":
        xb = xb[r.integers(0, 3, rows)]
    xb, xq = xb.astype(np.float32), xq.astype(np.float32)
    idx = hx.Index(d, 1, 1, 1)
    idx.set_centroids(xb[:1])
    idx.add(rows, xb)
    prm = hx.make_params(nprobe=1, algo=hx.ALGO_BATCHED, warmup_lists=1, warmup_list_size=1,
                         precision=hx.PREC_BF16 if data == "bf16" else hx.PREC_FP32)
    D, I, st = idx.search(n, xq, k, params=prm)
    assert st.survivors == n * rows and st.fallback_queries == 0
    m = min(n, 48)
    OD, OI, _ = oracle.Index.build(1, xb, xb[:1]).search(xq[-m:], 1, k)
    assert np.array_equal(I[-m:], OI) and np.array_equal(D[-m:].view(np.uint32), OD.view(np.uint32))


@pytest.mark.parametrize("data", ["int", "real"])
@pytest.mark.parametrize("n", [6, 3100])
@pytest.mark.parametrize("rows,over", [(512, False), (513, True), (700, True)])
def test_buffer_edge(rows, over, n, data):
    """A buffer of 512: exactly full, and one row more (the exact rescans)."""
    print(f"[case] {data} rows={rows} n={n} cap=512", flush=True)
    d, k = 12, 30
    r = np.random.default_rng(rows)
    xb, xq = (r.normal(0, 40, (m, d)) + 100 for m in (rows, n))
    if data == "int":
        xb, xq = (np.clip(np.rint(x), 0, 255) for x in (xb, xq))
    xb, xq = xb.astype(np.float32), xq.astype(np.float32)
    idx = hx.Index(d, 1, 1, 1)
    idx.set_centroids(xb[:1])
    idx.add(rows, xb)
    D, I, st = idx.search(n, xq, k, params=hx.make_params(nprobe=1, algo=hx.ALGO_BATCHED, warmup_lists=1,
                                                          warmup_list_size=1, survivor_cap=512))
    assert st.overflow_queries == (n if over else 0)
    m = min(n, 48)
    OD, OI, _ = oracle.Index.build(1, xb, xb[:1]).search(xq[-m:], 1, k)
    assert np.array_equal(I[-m:], OI) and np.array_equal(D[-m:].view(np.uint32), OD.view(np.uint32))
