"""The y forward pass's serial form, with the predictor's and corrector's
epilogues: the grids of more workgroups (of 16 columns) than it needs.

FP64 tiles that leave one workgroup to a CU (y lengths 144 and 192, and 128
unpadded) on grids of more than 256 workgroups, and FP32 tiles of 144 rows and
more above 384 workgroups.  One predict-and-correct and one further correction
against the FP64 oracle, and the carry form's passes against those.

Bars, FP64: 1e-12 relative L2, 1e-9 for the error (a sum of squares of
differences that lose up to three digits).  Mixed: the nonlinear term passes
about 44 radix-2 stages of FP32 transforms (three axes, there and back), each
adding at most 6e-8 of the RMS, in quadrature 4e-7, and a product whose factors
are a few times its RMS: 3e-6.  The velocity moves by dt / 2 of that, and by
|N| / |u| below 10: 1.5e-7.  The carry form evaluates the same increments: 1e-9.
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


@pytest.mark.parametrize("precision,nx,ny,nz,over", [
    ("fp64", 96, 128, 96, True), ("fp64", 96, 128, 96, False), ("fp64", 96, 96, 96, True),
    ("mixed", 128, 96, 128, True), ("mixed", 128, 128, 128, True)])
def test_step_against_oracle(precision, nx, ny, nz, over):
    from dnsjax_amd.fields import periodic_field
    from dnsjax_amd.flows import TriplyPeriodicFlow

    kw = dict(nx=nx, ny=ny, nz=nz, lx=L, ly=L, lz=L, re=40.0, dt=0.01, system="kolmogorov", oversample_y=over)
    assert (nz - 1) * -(-(nx // 2) // 16) > (256 if precision == "fp64" else 384)
    flow = TriplyPeriodicFlow(Params(precision=precision, tile_cols=16, **kw))
    nat = flow._native
    of = P.Flow(P.PeriodicParams(**kw))
    pc, ic = S.make_stepper(P.get_rhs, P.predict, P.correct, P.norm)
    u = periodic_field(nx, ny, nz, L, L, L, 0.1, 5)
    print(f"y forward, serial: {(nx, ny, nz)} {precision}", flush=True)
    d = flow.to_device(u)
    gp, gr, _ = flow.predict_and_correct(d)
    gp, gr, ge = flow.iterate_correction(d, gp, gr)
    cp, carry, ce = nat.empty(), nat.empty(), nat.scalar()
    nat.predict_and_correct_carry(d, cp, carry, ce)
    nat.iterate_correction_carry(cp, carry, ce)
    op, orr, _ = pc(u, of)
    op, orr, oe = ic(u, op, orr, of)
    fp64 = precision == "fp64"
    assert rel(gp, op) < (1e-12 if fp64 else 1.5e-7)
    assert rel(gr, orr) < (1e-12 if fp64 else 3e-6)
    assert rel(cp, gp.cpu().numpy()) < (1e-12 if fp64 else 1e-9)
    if fp64:
        assert abs(float(ge) - oe) < 1e-9 * oe and abs(float(ce) - oe) < 1e-9 * oe


@pytest.mark.parametrize("nx,ny,nz", [(16, 128, 16), (96, 96, 96)], ids=str)
def test_batched_members_equal_their_eager_runs(nx, ny, nz):
    """Members of a batch take the form of an eager run, on either side of the rule."""
    from dnsjax_amd.driver import run
    from dnsjax_amd.flows import TriplyPeriodicFlow
    from dnsjax_amd.native import BatchPlan

    def flow(i):
        return TriplyPeriodicFlow(Params(nx=nx, ny=ny, nz=nz, lx=L, ly=L, lz=L, re=40.0 + i, dt=0.01, tile_cols=16,
                                         system="kolmogorov", corrector_tolerance=1e-10, max_corrector_iterations=10))

    flows = [flow(i) for i in range(2)]
    states = [f.init_state(seed=70 + i, rms=0.05) for i, f in enumerate(flows)]
    refs = [run(flow(i), u.clone(), 1) for i, u in enumerate(states)]
    nats = [f._native for f in flows]
    nexts = [n.empty() for n in nats]
    counts = [torch.zeros(1, dtype=torch.int32, device=u.device) for u in states]
    plan = BatchPlan(nats, states, nexts, [n.empty() for n in nats], [n.empty() for n in nats], 10, counts=counts)
    plan.enqueue()
    torch.cuda.synchronize()
    for nxt, c, r in zip(nexts, counts, refs):
        assert torch.equal(nxt, r.state) and [int(c)] == r.counts
