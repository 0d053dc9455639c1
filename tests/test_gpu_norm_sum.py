"""The norm's final sum on either side of its two workgroup sizes.

The field's partial sums number ceil(modes / 256): 8 (fewer than a thread's
loads), 2017 (the last size of 256 threads' one round of loads, ragged) and
3025 (1024 threads, ragged).  Bar: 1e-13 relative, against the FP64 oracle's
norm; a sum of n positive terms in groups loses at most the depth of its
longest chain, below 40 roundings of 1.1e-16 per side.
"""

import math

import pytest

torch = pytest.importorskip("torch")

pytestmark = pytest.mark.gpu

from dnsjax_amd.params import Params  # noqa: E402
from oracle import periodic as P  # noqa: E402

L = 2 * math.pi


@pytest.fixture(scope="module", autouse=True)
def _gpu():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")


@pytest.mark.parametrize("shape", [(16, 16, 16), (64, 128, 128), (96, 128, 128)], ids=str)
def test_norm_against_oracle(shape):
    from dnsjax_amd.flows import TriplyPeriodicFlow

    nx, ny, nz = shape
    kw = dict(nx=nx, ny=ny, nz=nz, lx=L, ly=L, lz=L, re=40.0, dt=0.01, system="kolmogorov")
    flow = TriplyPeriodicFlow(Params(tile_cols=16, **kw))
    print(f"norm: {shape}", flush=True)
    g = torch.Generator().manual_seed(3)
    u = torch.randn(tuple(flow._native.shape), generator=g, dtype=torch.complex128)
    ref = P.norm(u.numpy(), P.Flow(P.PeriodicParams(**kw)))
    assert abs(float(flow.norm(flow.to_device(u.numpy()))) - ref) < 1e-13 * ref
