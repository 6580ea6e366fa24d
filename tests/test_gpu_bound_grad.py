"""The bound model's weight gradients (summed per chunk of rows, then over the
chunks) at the edges of their tiles and chunks.  Weights, inputs and dy are
small integers, so every FP32 sum is an integer below 2^24 and exact in any
order: the gradients equal the FP64 reference's bit for bit."""
import numpy as np
import pytest

from harmonyclient_amd import index as hx
from oracle import mlp_ref

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows,in_dim,hid", [
    (1, 33, 128), (31, 33, 64), (33, 33, 65), (1000, 5, 72), (2049, 33, 130), (4097, 70, 8), (300, 1, 1),
])
def test_integer_gradients_exact(rows, in_dim, hid):
    print(f"[case] gradient rows={rows} in={in_dim} hidden={hid}", flush=True)
    r = np.random.default_rng(rows + hid)
    p = r.integers(-1, 2, mlp_ref.num_params(in_dim, hid)).astype(np.float32)
    p[-2 * in_dim - 2:-in_dim - 2] = 0.0  # mu
    p[-in_dim - 2:-2] = 1.0               # sd
    p[-2:] = [1.0, 0.0]                   # scale, offset
    x = r.integers(-2, 3, (rows, in_dim)).astype(np.float32)
    dy = r.integers(-1, 2, rows).astype(np.float32)
    ref = mlp_ref.grad(p, x, dy, in_dim, hid)
    assert np.abs(ref).max() < 2 ** 24
    m = hx.TauModel(hidden=hid, in_dim=in_dim)
    m.set_params(p)
    for _ in range(2):  # (the second call reuses the workspaces)
        assert np.array_equal(m.grad(x, dy).astype(np.float64), ref)
    y = mlp_ref.forward(p, x, in_dim, hid)[0]
    assert np.array_equal(m.forward(x).astype(np.float64), y)
