"""A mixed plane Couette context's influence-matrix step, to the bit.

Every evaluation of a mixed context starts by rounding the iterate to FP32.  A
change in the iterate's last bit can round an element to the other neighbour:
1e-7 of the RMS in an element of the nonlinear term that a step returns.  So
the mixed form keeps one order of operations, and its results are compared with
recorded ones without a tolerance, for each stencil order, in the chunked solve
(five launches and one launch) and in the sequential sweeps.

golden/walls_mixed_bits.npz holds the corrected velocity of the inputs below on
gfx950, as plane Couette contexts gave it when the chunked solve broadcast each
window to one lane per map row (16-row chunks, one fused multiply-add per window
row in ascending order).  No other implementation pins these bits.
"""

import math
from pathlib import Path

import numpy as np
import pytest

torch = pytest.importorskip("torch")

pytestmark = pytest.mark.gpu

from dnsjax_amd.params import Params  # noqa: E402

GOLDEN = Path(__file__).parent / "golden" / "walls_mixed_bits.npz"
NX, NY, NZ = 8, 37, 8  # three chunks, the last of five rows


@pytest.fixture(scope="module", autouse=True)
def _gpu():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")


def field(seed):
    """Complex values in (-1/2, 1/2) from integer arithmetic alone."""
    shape = (3, NZ - 1, NX // 2, NY)
    i = np.arange(2 * np.prod(shape), dtype=np.uint64) + np.uint64(7919 * seed)
    i = (i * np.uint64(2654435761)) % np.uint64(1 << 32)
    i = ((i ^ (i >> np.uint64(13))) * np.uint64(1597334677)) % np.uint64(1 << 32)
    v = i.astype(np.float64) / 2.0**32 - 0.5
    return torch.from_numpy((v[0::2] + 1j * v[1::2]).reshape(shape)).cuda()


def corrected(p, variants):
    from dnsjax_amd.flows import PlaneCouetteFlow

    flow = PlaneCouetteFlow(Params(system="plane-couette", lx=2 * math.pi, lz=math.pi, nx=NX, ny=NY, nz=NZ, fd_order=p,
                                   re=400.0, dt=0.0123, implicitness=0.6, precision="mixed", tile_cols=16,
                                   variants=variants))
    out, _ = flow.correct(*(field(s) for s in (1, 2, 3, 4)))
    return out.cpu().numpy()


@pytest.mark.parametrize("form,variants", [("chunks", 0), ("chunks", 16), ("sweeps", 8)])
@pytest.mark.parametrize("p", [2, 4, 6, 8])
def test_mixed_step_keeps_its_bits(p, form, variants):
    want = np.load(GOLDEN)[f"{form}_{p}"]
    assert np.array_equal(corrected(p, variants), want)
