"""The MFMA coarse quantizer at every chunk count and around its groups of four
chunks, centroid counts around its 32-row tiles, query counts around 32, both
metrics, against the oracle's probes.  Lists and distances bit for bit."""
import numpy as np
import pytest

import oracle
from harmonyclient_amd import index as hx

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("metric", [0, 1])
@pytest.mark.parametrize("d", [1, 15, 16, 17, 33, 64, 65, 100, 112, 113, 128, 129, 145, 200, 256, 257, 420, 512])
@pytest.mark.parametrize("nlist,n", [(31, 33), (64, 64), (97, 1)])
def test_probes(metric, d, nlist, n):
    print(f"[case] metric={metric} d={d} nlist={nlist} n={n}", flush=True)
    r = np.random.default_rng(d + nlist)
    xb, xq, cent = (r.normal(0, 3, (m, d)).astype(np.float32) for m in (400, n, nlist))
    ix = oracle.Index.build(metric, xb, cent)
    idx = hx.Index(d, nlist, 1, metric)
    idx.set_centroids(cent)
    idx.add(400, xb)
    for P in (2, 20):
        OD, OI, _ = ix.search(xq, P, 7)
        D, I, _ = idx.search(n, xq, 7, params=hx.make_params(nprobe=P))
        assert np.array_equal(I, OI), f"{(I != OI).sum()} ids differ"
        assert np.array_equal(D.view(np.uint32), OD.view(np.uint32))
