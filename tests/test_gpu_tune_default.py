"""The autotuner keeps the built-in default where no candidate beats it (small
batches, whose default items hold fewer rows than any candidate's, and
real-valued lists past 128 dims, whose default is a form of its own): a tuned
index is never slower than the default it was compared with, and reports what
its searches then run."""
import numpy as np
import pytest

from harmonyclient_amd import index as hx

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("d,data", [(96, "real"), (200, "real"), (420, "real"), (128, "int")])
def test_default_is_a_candidate(d, data):
    import torch
    r = np.random.default_rng(d)
    rows, nlist, k = 60_000, 300, 10
    c = r.uniform(0, 255, (nlist, d))

    def points(m):
        x = c[r.integers(0, nlist, m)] + r.normal(0, 20, (m, d))
        return (np.clip(np.rint(x), 0, 255) if data == "int" else x).astype(np.float32)

    xb = points(rows)
    idx = hx.Index(d, nlist, 1, 1)
    idx.set_centroids(xb[:nlist])
    idx.add(rows, xb)
    for n, P in ((1, 4), (3, 16), (10, 8), (20, 24), (37, 24), (60, 30), (400, 16), (1500, 40)):
        print(f"[case] {data} d={d} n={n} P={P}", flush=True)
        xq = points(n)
        q = torch.from_numpy(xq).cuda()
        torch.cuda.synchronize()
        prm = hx.make_params(nprobe=P, algo=hx.ALGO_BATCHED)
        idx.set_tune()
        D0, I0, st0 = idx.search(n, xq, k, params=prm)
        t = idx.autotune(n, q.data_ptr(), k, params=prm, reps=5)
        print(f"[tune] {t}", flush=True)
        assert 0 < t["ms"] <= t["ms_default"]
        D, I, st = idx.search(n, xq, k, params=prm)
        assert np.array_equal(I, I0) and np.array_equal(D, D0)
        assert (st.batch_queries, st.batch_rows, st.batch_waves) == (t["batch_queries"], t["batch_rows"], t["batch_waves"])
        if t["ms"] == t["ms_default"]:
            assert (st.batch_queries, st.batch_rows, st.batch_waves) == (st0.batch_queries, st0.batch_rows, st0.batch_waves)
