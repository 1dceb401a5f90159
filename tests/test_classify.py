"""Coarse flags and neighbour masks (updateFields, pressure_solver.hpp:40-57)
computed several levels a launch, against the oracle: every level's flags,
and the masks through two V-cycles, bit-identical.  Sizes on both sides of a
64-cell tile and its coarsenings, of the one-workgroup tail (16384
cells), hierarchies of 2 to 10 levels and elongated ones; the
allocation-free solve on top, with flag bytes other than 0 and 1, whose
scratch holds the contents of the call before."""
import numpy as np
import pytest

import ubootgl_amd as U
from oracle import pyoracle as O
from test_zz_no_alloc import _noalloc

pytestmark = pytest.mark.gpu

SIZES = [(1100, 900), (8, 8), (9, 17), (128, 128), (129, 128), (127, 131), (191, 193), (65, 2050),
         (513, 64), (1000, 130), (2049, 16), (4200, 9), (449, 385)]


@pytest.mark.parametrize("W,H", SIZES)
def test_flags_and_masks(gpu, W, H):
    g = np.random.default_rng(W * 7 + H)
    flag = (g.random((H, W)) < g.choice([0.1, 0.3, 0.85])).astype(np.float32)
    f = g.standard_normal((H, W)).astype(np.float32)
    p = g.standard_normal((H, W)).astype(np.float32)
    h = float(np.float32(1.0 / W))
    mg, om = U.MG(flag), O.OracleMG(W, H)
    om.update_fields(flag)
    for l in range(len(om.sizes)):
        np.testing.assert_array_equal(mg.get_flag(l), om.flag_level(l), err_msg=f"level {l}")
    got, want = p.copy(), p.copy()
    for _ in range(2):
        mg.solve(got, f, flag, h, True)
        om.solve(want, f, flag, h, True)
    np.testing.assert_array_equal(got, want)
    mg.close()
    np.testing.assert_array_equal(_noalloc(p, f, flag * 255, h, 1, 2), want)
