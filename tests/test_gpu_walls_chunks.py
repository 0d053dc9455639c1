"""The matrix-core band solves of the influence-matrix step at the edges of
their chunks (8 to 20 new rows in windows of 16 or 32), of the 64-row groups of
points per lane, and at the shortest and longest columns of the one-launch form.

The sequential sweeps solve the same systems (LU with the reference's order of
operations).  Both are backward stable; they are held together at 1e-11
relative L2, ten times the bar each is held to against the FP64 oracle."""

import math

import numpy as np
import pytest

torch = pytest.importorskip("torch")

pytestmark = pytest.mark.gpu

from dnsjax_amd.params import Params  # noqa: E402


@pytest.fixture(scope="module", autouse=True)
def _gpu():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")


def native(nx, ny, nz, p, variants):
    from dnsjax_amd.flows import PlaneCouetteFlow

    return PlaneCouetteFlow(Params(system="plane-couette", lx=2 * math.pi, lz=math.pi, nx=nx, ny=ny, nz=nz,
                                   fd_order=p, re=400.0, dt=0.01, tile_cols=16, variants=variants))._native


@pytest.mark.parametrize("p", [2, 4, 6, 8])
@pytest.mark.parametrize("ny", ["least", 16, 17, 32, 33, 64, 65, 80, 128, 129, 240, 256, 257, 278])
def test_forms_agree_at_chunk_edges(ny, p):
    nx, nz = 8, 8  # (7, 4) modes: k^2 classes of one and of two
    ny = p + 5 if ny == "least" else ny
    from dnsjax_amd.fields import wall_field

    g = torch.Generator().manual_seed(ny + p)
    u = torch.as_tensor(wall_field(nx, ny, nz, 2 * math.pi, math.pi, 0.1, seed=ny)).cuda()
    n = torch.randn(u.shape, dtype=torch.complex128, generator=g).cuda()
    out = {v: native(nx, ny, nz, p, v).predict(u, n) for v in (0, 8, 16)}
    assert torch.equal(out[0], out[16])
    d = float(torch.linalg.norm(out[16] - out[8]) / torch.linalg.norm(out[8]))
    assert d < 1e-11, d


@pytest.mark.parametrize("variants", [0, 16])
def test_a_bad_mode_stays_alone(variants):
    """NaN in one mode's state does not reach the mode that shares its workgroup."""
    nx, ny, nz, p = 8, 33, 8, 6
    nat = native(nx, ny, nz, p, variants)
    g = torch.Generator().manual_seed(1)
    u = torch.randn((3, nz - 1, nx // 2, ny), dtype=torch.complex128, generator=g).cuda()
    n = torch.randn(u.shape, dtype=torch.complex128, generator=g).cuda()
    good = nat.predict(u, n)
    u[1, 1, 1, ny - 1] = float("nan")  # its class partner is the mode of -kz, (nz - 2, 1)
    bad = nat.predict(u, n)
    keep = np.ones((nz - 1, nx // 2), bool)
    keep[1, 1] = False
    assert torch.isnan(bad[:, 1, 1].real).any()
    assert torch.equal(bad[:, keep], good[:, keep])
