"""Chunked band solves of the columns past the one-launch form's, up to the
longest that their LDS rows take, and the limits of both forms.

641 has the most zero rows behind the last chunk of order 8 and mixed contexts
(65392 bytes of LDS).  Held to the sequential sweeps as the columns up to 278
are (1e-11 relative L2), with four times their bar: two FP64 solutions of these
systems on the CPU (banded and dense LU) differ by 0.3e-12 to 1.2e-12 at 278
points and by 1e-12 to 3e-12 at 641."""

import math

import pytest

torch = pytest.importorskip("torch")

pytestmark = pytest.mark.gpu

from dnsjax_amd.params import Params  # noqa: E402


@pytest.fixture(scope="module", autouse=True)
def _gpu():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")


def native(ny, p, variants, precision="fp64"):
    from dnsjax_amd.flows import PlaneCouetteFlow

    return PlaneCouetteFlow(Params(system="plane-couette", lx=2 * math.pi, lz=math.pi, nx=8, ny=ny, nz=8, fd_order=p,
                                   re=400.0, dt=0.01, tile_cols=16, variants=variants, precision=precision))._native


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("p", [2, 4, 6, 8])
@pytest.mark.parametrize("ny", [279, 320, 512, 641, 649, 650])
def test_long_columns_agree_with_the_sweeps(ny, p, precision):
    from dnsjax_amd.fields import wall_field

    g = torch.Generator().manual_seed(ny + p)
    u = torch.as_tensor(wall_field(8, ny, 8, 2 * math.pi, math.pi, 0.1, seed=ny)).cuda()
    n = torch.randn(u.shape, dtype=torch.complex128, generator=g).cuda()
    a, b = (native(ny, p, v, precision).predict(u, n) for v in (0, 8))
    assert float(torch.linalg.norm(a - b) / torch.linalg.norm(b)) < 4e-11


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_limits(precision):
    u = torch.zeros((3, 7, 4, 279), dtype=torch.complex128, device="cuda")
    nat = native(279, 4, 16, precision)
    with pytest.raises(Exception, match="fused form"):
        nat.predict(u, u)
    with pytest.raises(Exception, match="chunk maps exceed"):
        native(651, 4, 0, precision)
    native(651, 4, 8, precision)
