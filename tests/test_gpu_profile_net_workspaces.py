"""The profile network's entry points take NULL for the work arguments that no
kernel uses: `part` of the gradient, `wf` of the forward pass and of the guess;
the wrapper allocates none of them."""

import math

import pytest

torch = pytest.importorskip("torch")

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def _gpu():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")


def test_unused_workspaces_may_be_null():
    from dnsjax_amd import _lib, profile_net

    net = profile_net.ProfileNet(17, 64, seed=3)
    B = 70
    g = torch.Generator().manual_seed(4)
    X = torch.randn((B, net.din), generator=g).bfloat16().view(torch.int16).cuda()
    T = torch.randn((B, net.dout), generator=g).cuda()
    Y, loss = net.forward(X), float(net.compute_grad(X, T))
    grad = net.grad.clone()
    wb, wh = torch.zeros_like(net.wb), torch.zeros(B * (3 * net.H + net.dout), dtype=torch.int16, device="cuda")
    wf = torch.zeros(B * (2 * net.H + net.dout), device="cuda")
    y, gr, ls = torch.zeros_like(Y), torch.zeros_like(grad), torch.zeros((), device="cuda")
    s = torch.cuda.current_stream().cuda_stream
    size = (net.din, net.H, net.dout, B)
    _lib.check(net.lib.dnsmi_pnet_forward(*size, X.data_ptr(), net.params.data_ptr(), wb.data_ptr(), None,
                                          wh.data_ptr(), y.data_ptr(), s))
    _lib.check(net.lib.dnsmi_pnet_grad(*size, X.data_ptr(), T.data_ptr(), net.params.data_ptr(), wb.data_ptr(),
                                       wf.data_ptr(), wh.data_ptr(), None, gr.data_ptr(), ls.data_ptr(), s))
    torch.cuda.synchronize()
    assert torch.equal(y, Y) and torch.equal(gr, grad) and float(ls) == loss


def test_the_wrapper_allocates_no_unused_workspace():
    from dnsjax_amd import profile_net
    from dnsjax_amd.flows import PlaneCouetteFlow
    from dnsjax_amd.learned import Scales
    from dnsjax_amd.params import Params

    flow = PlaneCouetteFlow(Params(system="plane-couette", lx=2 * math.pi, lz=math.pi, nx=16, ny=17, nz=16, re=400.0,
                                   dt=0.01))
    nat = flow._native
    u = flow.init_state(seed=1, rms=0.05)
    n0 = nat.get_rhs(u)
    h = [torch.view_as_real(n0).float().contiguous() for _ in range(2)]
    net = profile_net.ProfileNet(17, 64, seed=3)
    pred, rhs = nat.empty(), nat.empty()
    net.guess(nat, u, pred, rhs, h[0], h[1], Scales(1.0, 1.0, 0.1))
    torch.cuda.synchronize()
    assert torch.isfinite(torch.view_as_real(pred)).all()
    assert set(net._work) == {"gX", "gwh", "gY"}
