"""The weight gradients' split of a batch: no part without samples.

At (32 -> 128 -> 128 -> 200) and 6700 samples the output layer's gradient is
split into parts of three chunks of 64 samples, of which the batch fills 35.
The parts lie one behind the other in the work buffer; a part without samples
would be launched, stored as zeros and summed.
"""

import pytest

torch = pytest.importorskip("torch")

pytestmark = pytest.mark.gpu


def test_no_part_is_empty():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from dnsjax_amd import _lib

    din, H, dout, B = 32, 128, 200, 6700
    lib = _lib.load()
    g = torch.Generator().manual_seed(5)
    n = din * H + H + H * H + H + H * dout + dout
    prm = (0.1 * torch.randn(n, generator=g)).cuda()
    X = torch.randn((B, din), generator=g).bfloat16().cuda()
    T = torch.randn((B, dout), generator=g).cuda()
    wb = torch.zeros(n, dtype=torch.int16, device="cuda")
    wf = torch.full((B * (2 * H + dout),), float("nan"), device="cuda")
    wh = torch.zeros(B * (3 * H + dout), dtype=torch.int16, device="cuda")
    part = torch.zeros(B * dout // 256 + 1, device="cuda")
    grad, loss = torch.zeros(n, device="cuda"), torch.zeros((), device="cuda")
    _lib.check(lib.dnsmi_pnet_grad(din, H, dout, B, X.data_ptr(), T.data_ptr(), prm.data_ptr(), wb.data_ptr(),
                                   wf.data_ptr(), wh.data_ptr(), part.data_ptr(), grad.data_ptr(), loss.data_ptr(),
                                   torch.cuda.current_stream().cuda_stream))
    torch.cuda.synchronize()
    assert torch.isfinite(grad).all() and torch.isfinite(loss)
    size = (H + 1) * dout  # one part of the output layer's gradient: H rows and the bias's
    parts = wf[2 * B * H:]
    parts = parts[:parts.numel() // size * size].view(-1, size)
    assert not (parts == 0).all(1).any()
