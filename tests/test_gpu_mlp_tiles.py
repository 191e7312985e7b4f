"""The network's tiled products (32 x 64 tiles, k in chunks of 64, the batch in
ranges of at least 128 rows) at sizes on and beside those edges, against the
FP64 oracle.

Tolerance: every product sums at most a few thousand FP32 terms of the batch
(relative error of a sum of n terms below n eps in the worst case, about
sqrt(n) eps for these), through three layers; 5e-5 of the largest gradient
entry is above 8 * sqrt(5000) * 6e-8.
"""
import numpy as np
import pytest

from oracle import mlp_oracle as M

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nin,nemb,nmodes,nhid,N", [
    (1, 0, 1, 1, 1),          # nothing but edges, no embedding
    (64, 0, 2, 64, 64),       # whole tiles and chunks
    (48, 16, 16, 32, 129),    # one row past a range
    (33, 64, 16, 65, 127),    # one past a tile, the widest embedding table
    (120, 3, 5, 130, 1025),
    (128, 16, 3, 300, 5000),  # more tiles than ranges
])
def test_tile_edges(hip, nin, nemb, nmodes, nhid, N):
    from mlcp_amd.warmstart import MLP
    print("[case] mlp tiles", nin, nemb, nmodes, nhid, N, flush=True)
    rng = np.random.default_rng(nin + N)
    net = MLP(nin, nmodes, nemb=nemb, nhid=nhid, seed=1)
    p = rng.normal(scale=0.5 / np.sqrt(nhid), size=net.np).astype(np.float32)
    net.set_params(p)
    X = rng.normal(size=(N, nin)).astype(np.float32)
    X /= np.linalg.norm(X, axis=1, keepdims=True)
    T = rng.normal(size=(N, nin)).astype(np.float32)
    modes = rng.integers(0, nmodes, size=N).astype(np.int32)
    dims = (nin, nemb, nmodes, nhid)
    loss, g = net.loss_grad(X, modes, T)
    lo, go = M.loss_grad(p.astype(np.float64), X, modes, T, *dims)
    assert abs(loss - lo) <= 1e-5 * abs(lo)
    assert np.max(np.abs(g - go)) <= 5e-5 * np.abs(go).max()
    Y = net.forward(X, modes)
    Yo = M.forward(p.astype(np.float64), X, modes, *dims)
    assert np.max(np.abs(Y - Yo)) <= 1e-5 * np.abs(Yo).max()
