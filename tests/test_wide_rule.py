"""The step's per-cell passes on both sides of the rule that takes them to wide
rows, bit-identical to the oracle's step: fields of 5 strips (diffuse only) and of
9 and 13 (all passes) that end with, one and three cells past a whole strip, one
strip fewer, and heights whose bands are whole, nearly whole and too uneven."""
import pytest

from ubootgl_amd import workloads
from oracle import pyoracle as O
from test_gpu_parity import FIELDS, compare, make_pair

pytestmark = pytest.mark.gpu

# a strip owns 124 columns of the W - 1 from column 1; four rows a block (eight
# for diffuse), 32 blocks a band of all XCDs
CASES = [(497, 18201), (621, 14595), (622, 14594), (624, 14593),      # 4 and 5 strips
         (993, 9071), (1117, 8101), (1118, 8102), (1120, 8100),       # 8 and 9
         (1489, 6147), (1613, 5634), (1614, 5635), (1616, 5633),      # 12 and 13
         (8933, 1026), (8934, 1027), (8700, 1100), (12901, 701), (17001, 561), (60001, 161)]


@pytest.mark.parametrize("W,H", CASES)
def test_step_on_both_sides(gpu, W, H):
    k = W + H
    d = workloads.small_domain(W, H, seed=k, ndisks=9)
    sim, ref = make_pair(d)
    bcs = [(k >> i) % 4 for i in range(4)]
    sim.setBCs(*bcs)
    ref.set_bcs(*bcs)
    sim.step(float(d.dt))
    ref.step(float(d.dt))
    compare(sim, ref, FIELDS + [("vx_current", O.VX_CURRENT), ("vy_current", O.VY_CURRENT)])
