"""Values that overflow in a level pass (a source (f h) h beyond the largest
float, four times a pressure beyond it): the pass gives what the stand-alone
sweeps and grid transfers give, NaN for NaN, whether the cell's row is all
fluid or holds an obstacle elsewhere, in every tile shape.  Two levels of the
hierarchy are solved and the coarse one takes no sweep, so that nothing but the
passes of level 0 reaches its pressure."""
import numpy as np
import pytest

import ubootgl_amd as U
from ubootgl_amd import _lib as L

pytestmark = pytest.mark.gpu

H = 29  # 29, 14 and 7 rows: level 1 is the coarsest solved
# 12 and 16 waves of 2 rows, 8 of 4, 8 of 6
WIDTHS = [400, 30300, 60000, 150000]


@pytest.mark.parametrize("zg", [False, True])
@pytest.mark.parametrize("pre,post", [(0, 0), (0, 1), (1, 2), (3, 3)])
@pytest.mark.parametrize("W", WIDTHS)
def test_overflow_as_stand_alone(gpu, W, pre, post, zg):
    g = np.random.default_rng(W)
    flag = np.ones((H, W), np.float32)
    f = np.zeros((H, W), np.float32)
    p = g.standard_normal((H, W)).astype(np.float32)
    flag[14, 60::128] = 0  # rows 13 to 15 of some tiles are not uniform
    for k, x in enumerate(range(30, W - 30, 97)):
        for y in (5 + k % 2, 14, 22):
            f[y, x] = 3.3e38 * (-1) ** k
        # four times the middle overflows, the sum of its neighbours does not
        p[9, x + 9:x + 12] = p[8:11, x + 10] = 0.8e38
        p[9, x + 10] = 1e38
    h = 1.05
    m = U.MG(flag)
    m.set_params(U.Params(nu_pre=pre, nu_post=post, nu_coarse=0))
    m.set_level(0, 0, p)
    m.set_level(0, 1, f)
    m.solve_resident(h, zg, 1)
    got = m.get_level(0, 0), m.get_level(1, 1)
    m.set_level(0, 0, p)

    def sweeps(n):
        for _ in range(n):
            m.level_op(L.MGOP_RBGS, 0, h)
            if zg:
                m.level_op(L.MGOP_ZERO_GRADIENT, 0, h)

    sweeps(pre)
    m.level_op(L.MGOP_RESTRICT_RESIDUAL, 0, h)
    m.level_op(L.MGOP_PROLONG_CORRECT, 0, h)
    if zg:
        m.level_op(L.MGOP_ZERO_GRADIENT, 0, h)
    sweeps(post)
    want = m.get_level(0, 0), m.get_level(1, 1)
    m.close()
    assert np.isnan(want[0]).any() or post == 0
    assert not np.isfinite(want[1]).all()
    for a, b in zip(got, want):
        np.testing.assert_array_equal(a, b)
