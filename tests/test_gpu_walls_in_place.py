"""The influence-matrix step in place: the predictor's output may be its state,
a corrector's output its iterate.  Every form, in a box with a k^2 class of an
odd number of modes (one of its workgroups repeats its first mode)."""

import math

import pytest

torch = pytest.importorskip("torch")

pytestmark = pytest.mark.gpu

from dnsjax_amd.params import Params  # noqa: E402

NX, NY, NZ = 16, 65, 16


@pytest.fixture(scope="module", autouse=True)
def _gpu():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("variants", [0, 8, 16])
@pytest.mark.parametrize("p", [4, 8])
def test_in_place_equals_out_of_place(p, variants, precision):
    from dnsjax_amd.flows import PlaneCouetteFlow

    nat = PlaneCouetteFlow(Params(system="plane-couette", lx=2 * math.pi, lz=math.pi, nx=NX, ny=NY, nz=NZ, fd_order=p,
                                  re=400.0, dt=0.01, tile_cols=16, variants=variants, precision=precision))._native
    g = torch.Generator().manual_seed(p)
    u, v, n, m = (torch.randn((3, NZ - 1, NX // 2, NY), dtype=torch.complex128, generator=g).cuda() for _ in range(4))
    want = nat.predict(u, n)
    w = u.clone()
    assert torch.equal(nat.predict(w, n, out=w), want) and torch.equal(w, want)
    want, corr = nat.correct(u, v, n, m)
    w = v.clone()
    out, got = nat.correct(u, w, n, m, out=w)
    assert torch.equal(out, want) and torch.equal(got, corr)
