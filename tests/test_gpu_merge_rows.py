"""Merges of short rows (one wave per query) at the edges of that form --
entries a lane holds, k kept, sort sizes -- with many equal distances, equal
entries and padding, against the oracle's merge bit for bit."""
import numpy as np
import pytest

import oracle
from conftest import random_partials
from harmonyclient_amd import index as hx

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("parts,k_in,k", [(1, 1, 1), (1, 64, 64), (2, 128, 256), (4, 64, 65), (257, 1, 100), (3, 171, 128),
                                          (8, 64, 129), (8, 100, 100), (7, 146, 256), (1, 1024, 256), (1024, 1, 33),
                                          (1024, 1, 257), (25, 41, 10)])
@pytest.mark.parametrize("metric", [hx.METRIC_L2, hx.METRIC_IP])
def test_short_rows(parts, k_in, k, metric):
    print(f"[case] {parts} x {k_in} k={k} metric={metric}", flush=True)
    n = 21
    Dp, Ip = random_partials(parts + k, parts, n, k_in, metric, ties=True)
    Dp[:, 1] = 2.0  # one distance only
    Dp[:, 2], Ip[:, 2] = -1.5, 7  # one entry, everywhere
    Ip[:, 3] = -1  # padding only
    Dp[:, 4] *= -1
    D, I = hx.merge_topk(metric, Dp, Ip, k)
    OD, OI = oracle.merge(metric, Dp, Ip, k)
    assert np.array_equal(I, OI), f"{(I != OI).sum()} ids differ"
    OD = OD + np.float32(0)  # a key holds +0 for -0
    assert np.array_equal(D.view(np.uint32), OD.view(np.uint32))
