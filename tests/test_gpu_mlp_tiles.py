"""The per-mode network's training gradient at the edges of its tiles: one
sample, a whole tile, one past it, and more tiles than workgroups (each then
takes several), against the FP64 oracle.
"""

import numpy as np
import pytest

torch = pytest.importorskip("torch")

pytestmark = pytest.mark.gpu

from oracle import mlp as M  # noqa: E402
from tests.test_gpu_learned import _net_with, _random_params, rel  # noqa: E402


@pytest.mark.parametrize("H", [32, 64])
@pytest.mark.parametrize("B", [1, 32, 33, 32 * 1024 + 45])
def test_gradient_tiles_match_oracle(H, B):
    rng = np.random.default_rng(B)
    params = _random_params(H, 11)
    x = rng.standard_normal((B, 16)).astype(np.float32).astype(np.float64)
    t = rng.standard_normal((B, 6)).astype(np.float32).astype(np.float64)
    loss, grads = M.loss_and_grads(params, x, t)
    net = _net_with(H, params)
    X, T = (torch.from_numpy(a).float().to(net.device) for a in (x, t))
    got_loss = float(net.compute_grad(X, T, bf16=False))
    assert abs(got_loss - loss) <= 1e-5 * loss
    first = net.grad.clone()
    o = 0
    for g in grads:
        assert rel(first[o:o + g.size].cpu().double().numpy(), g.reshape(-1)) <= 1e-4, o
        o += g.size
    net.compute_grad(X, T, bf16=False)
    assert torch.equal(net.grad, first)  # fixed-order sums
