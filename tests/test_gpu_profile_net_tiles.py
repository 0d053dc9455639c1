"""The profile network's matrix-core products at the edges of their tiles:
forward and every gradient against the oracle where rows, columns or the
contraction end inside a tile, a 64-deep chunk or a 16-byte load, and the
independence of an output from the batch (and so the tile) it is computed in.
"""

import numpy as np
import pytest

torch = pytest.importorskip("torch")

pytestmark = pytest.mark.gpu

from oracle import mlp as M  # noqa: E402
from tests.test_gpu_profile_net import _bf16_words, _net, _split, rel  # noqa: E402


# (din, H, dout, B): one sample and one output; columns narrower than a tile
# (odd, so that rows start at odd 2-byte addresses); rows and columns one past
# a tile; an odd number of 32-deep halves of a chunk; a batch split into
# several parts with a ragged last one; the large tile of a layer
@pytest.mark.parametrize("din,H,dout,B", [(32, 64, 1, 1), (32, 64, 63, 31), (96, 64, 65, 33), (160, 128, 129, 65),
                                          (64, 192, 130, 129), (608, 256, 451, 640), (32, 128, 200, 6700)])
def test_tile_edges_match_the_oracle(din, H, dout, B):
    net, params = _net(din, H, dout, seed=din + dout)
    rng = np.random.default_rng(B)
    x = M.to_bf16(rng.standard_normal((B, din)))
    t = rng.standard_normal((B, dout)) * 0.5
    X, T = _bf16_words(x), torch.from_numpy(t.astype(np.float32)).cuda()
    y_ref, _ = M.forward(params, x, bf16=True)
    assert rel(net.forward(X), y_ref) < 1e-3
    loss = net.compute_grad(X, T)
    want_loss, want = M.profile_loss_and_grads(params, x, t.astype(np.float32).astype(np.float64), bf16=True)
    assert abs(float(loss) - want_loss) <= 1e-3 * want_loss
    errs = [rel(a.double(), b) for a, b in zip(_split(net.grad, din, H, dout), want)]
    assert max(errs) < 2e-2, errs


@pytest.mark.parametrize("dout", [384, 385])
def test_outputs_do_not_depend_on_the_batch(dout):
    """Every output is one ascending accumulation over k in either tile."""
    net, _ = _net(1056, 128, dout, seed=5)
    X = _bf16_words(np.random.default_rng(3).standard_normal((13400, 1056)))
    Y = net.forward(X)
    for lo, n in ((0, 1), (100, 333), (13399, 1)):
        assert torch.equal(net.forward(X[lo:lo + n].contiguous()), Y[lo:lo + n])
