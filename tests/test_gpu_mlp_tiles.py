"""The network's gradient at the edges of its 16-sample tiles and of its 256
blocks, against the float64 oracle.

Tolerance: as in the learned-indicator tests, 1e-3 normwise (1e-4 for the loss)
over many samples; with few samples a single activation that rounds to the other
BF16 neighbour is not averaged out: one of 64 activations changed by 2^-8 moves
a gradient by 2^-8 / sqrt(64) = 5e-4 of its norm, a few such ones 5e-3."""
import numpy as np
import pytest

import goal_amd as g
from oracle import learned as L
from tests.test_gpu_learned import _net

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 15, 16, 17, 100, 4095, 4096, 4097, 8200])
def test_gradient_at_tile_edges(n):
    params, norms, X, Y = _net(11)
    mlp = g.MLP()
    mlp.set(params, norms)
    idx = np.random.default_rng(n).integers(0, X.shape[0], n).astype(np.int32)
    xd, yd = g.DeviceBuffer.from_host(X.ravel(), np.float32), g.DeviceBuffer.from_host(Y, np.float32)
    loss, grad = mlp.gradient(xd, yd, g.DeviceBuffer.from_host(idx, np.int32), n)
    rl, rg = L.mlp_loss_grad(params, norms, X[idx], Y[idx])
    few = n < 1000
    assert abs(loss - rl) <= (5e-3 if few else 1e-4) * rl
    assert np.linalg.norm(grad - rg) <= (5e-3 if few else 1e-3) * np.linalg.norm(rg)
