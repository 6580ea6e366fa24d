"""The form of plain batches with few probes: more queries do not take a faster form
and less time than fewer, nor half of them far less than half."""
import numpy as np
import pytest

from harmonyclient_amd import index as hx

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("d,nlist,rows,P,few,many,lo,hi", [
    (201, 16, 1250, 1, 4000, 8000, 1.45, 3.0), (201, 64, 1000, 1, 4000, 8000, 1.45, 3.0),
    (420, 16, 3000, 2, 125, 250, 0.8, 2.4), (420, 64, 3000, 2, 125, 250, 0.8, 2.4),
])
def test_time_grows_with_the_queries(d, nlist, rows, P, few, many, lo, hi):
    print(f"[case] d={d} nlist={nlist} rows={rows} P={P}", flush=True)
    r = np.random.default_rng(d + nlist)
    c = r.integers(0, 256, (nlist, d)).astype(np.float32)

    def near(l, s):
        return np.clip(np.rint(c[l] + r.normal(0, s, (len(l), d))), 0, 255).astype(np.float32)

    idx = hx.Index(d, nlist, P, 1)
    idx.set_centroids(c)
    idx.set_lists(np.arange(nlist + 1) * rows, np.arange(nlist * rows), near(np.repeat(np.arange(nlist), rows), 5))
    q = near(r.integers(0, nlist, many), 20)
    x, k = torch.from_numpy(q).cuda(), 10
    D = torch.empty(many, k, device="cuda")
    I = torch.empty(many, k, dtype=torch.int64, device="cuda")
    prm = hx.make_params(nprobe=P)
    _, pr = idx.coarse(q, P)
    SD, SI, _ = idx.scan(q, pr, k)
    ms = {}
    for n in (few, many):
        torch.cuda.synchronize()
        t = [idx.search_device(n, x.data_ptr(), k, D.data_ptr(), I.data_ptr(), prm, stats=True).total_ms for _ in range(9)]
        torch.cuda.synchronize()
        assert np.array_equal(I[:n].cpu().numpy(), SI[:n]) and np.array_equal(D[:n].cpu().numpy(), SD[:n])
        ms[n] = min(t)
    print(f"[time] {few} queries {ms[few] * 1e3:.0f} us, {many} {ms[many] * 1e3:.0f} us", flush=True)
    assert lo * ms[few] < ms[many] < hi * ms[few]
