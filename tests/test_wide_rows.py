"""The step's per-cell passes on wide rows (two cells a lane, large fields)
bit-identical to the oracle's step, at the sizes where a strip can go wrong:
domains narrower than a strip, a last strip that ends at, one before or one
past the domain's edge columns, odd and even row counts, and every
boundary-condition kind on every side.  The sizes straddle the passes'
thresholds: the first takes wide rows in the divergence only, the second in
the correction too, the others in all three."""
import pytest

from ubootgl_amd import workloads
from oracle import pyoracle as O
from test_gpu_parity import FIELDS, compare, make_pair

pytestmark = pytest.mark.gpu

CASES = [(41, 62001, (0, 1, 3, 2)), (84, 61003, (1, 0, 1, 3)), (249, 36501, (3, 3, 0, 0)),
         (250, 36402, (2, 2, 2, 1)), (252, 36001, (0, 2, 3, 3)), (3012, 2993, (0, 1, 3, 2))]


@pytest.mark.parametrize("W,H,bcs", CASES)
def test_wide_step(gpu, W, H, bcs):
    d = workloads.small_domain(W, H, seed=W + H, ndisks=12)
    sim, ref = make_pair(d)
    sim.setBCs(*bcs)
    ref.set_bcs(*bcs)
    for _ in range(2):
        sim.step(float(d.dt))
        ref.step(float(d.dt))
    compare(sim, ref, FIELDS + [("vx_current", O.VX_CURRENT), ("vy_current", O.VY_CURRENT)])
