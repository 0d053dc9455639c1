"""The y forward pass with its fused projection and update, both forms.

One predict-and-correct and one further correction against the FP64 oracle's
step, for column tiles of 8 and 16, partly filled tiles (nx / 2 no multiple of
the tile), the shortest and longest lengths, an unpadded y axis, and, at the
two lengths whose FP64 tile leaves one workgroup to a CU, grids on either side
of one workgroup per CU (96^3: 285 workgroups of 16 columns).  Bars: relative
L2 1e-12 for the FP64 fields and 1e-5 for the mixed ones (FP32 transforms),
relative 1e-9 for the FP64 corrector error (a sum of squares of differences
that lose up to three digits to cancellation).
"""

import math

import numpy as np
import pytest

torch = pytest.importorskip("torch")

pytestmark = pytest.mark.gpu

from dnsjax_amd.params import Params  # noqa: E402
from oracle import periodic as P  # noqa: E402
from oracle import stepper as S  # noqa: E402

L = 2 * math.pi


@pytest.fixture(scope="module", autouse=True)
def _gpu():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")


def rel(a, b):
    a = a.detach().cpu().numpy()
    return float(np.linalg.norm(a - b) / np.linalg.norm(b))


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("tile", [8, 16])
@pytest.mark.parametrize("shape", [
    (8, 8, 8, True), (16, 16, 8, True), (48, 32, 16, True), (32, 48, 16, True), (16, 64, 32, True),
    (32, 96, 16, True), (96, 96, 96, True), (32, 128, 48, True), (16, 16, 16, False), (48, 64, 8, False),
    (8, 128, 16, False)], ids=str)
def test_step_against_oracle(shape, tile, precision):
    from dnsjax_amd.fields import periodic_field
    from dnsjax_amd.flows import TriplyPeriodicFlow

    nx, ny, nz, over = shape
    kw = dict(nx=nx, ny=ny, nz=nz, lx=L, ly=L, lz=L, re=40.0, dt=0.01, system="kolmogorov", oversample_y=over)
    flow = TriplyPeriodicFlow(Params(precision=precision, tile_cols=tile, **kw))
    of = P.Flow(P.PeriodicParams(**kw))
    pc, ic = S.make_stepper(P.get_rhs, P.predict, P.correct, P.norm)
    u = periodic_field(nx, ny, nz, L, L, L, 0.1, 5)
    print(f"y forward: {shape} tile {tile} {precision}", flush=True)
    d = flow.to_device(u)
    gp, gr, _ = flow.predict_and_correct(d)
    gp, gr, ge = flow.iterate_correction(d, gp, gr)
    op, orr, _ = pc(u, of)
    op, orr, oe = ic(u, op, orr, of)
    bar = 1e-12 if precision == "fp64" else 1e-5
    assert rel(gp, op) < bar
    assert rel(gr, orr) < bar
    if precision == "fp64":
        assert abs(float(ge) - oe) < 1e-9 * oe
