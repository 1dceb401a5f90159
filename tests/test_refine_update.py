"""The refinement update (refine_device.hpp) where its columns and rows can go
wrong: widths on both sides of a wave (64) and of a block (256), heights on
both sides of a block's 8 rows, a random start and obstacles.  ||r|| before
and after one step against the float64 oracle's residual of the very x the
solver holds, and the batched update against the single one, bit for bit.

Tolerance: the norms differ by the order of at most 2^18 positive float64
terms, so by less than 2^18 eps = 6e-11 relative; a wrong cell moves them by
1e-6 or more."""
import numpy as np
import pytest

import ubootgl_amd as U
from ubootgl_amd.batch import Batch
from oracle import pyoracle as O

pytestmark = pytest.mark.gpu

SIZES = [(8, 8), (63, 9), (64, 15), (65, 16), (66, 17), (128, 24), (129, 31), (255, 33), (256, 40),
         (257, 41), (258, 8), (513, 130), (1000, 57)]


def problem(W, H):
    g = np.random.default_rng(W * 3 + H)
    flag = np.ones((H, W), np.float32)
    flag[1:-1, 1:-1] = g.random((H - 2, W - 2)) > 0.1
    f = g.standard_normal((H, W)).astype(np.float32)
    return flag, f, g.standard_normal((H, W)), float(np.float32(1.0 / W))


@pytest.mark.parametrize("W,H", SIZES)
def test_update_norms(gpu, W, H):
    flag, f, x0, h = problem(W, H)
    mg = U.MG(flag)
    mg.ir_set_rhs(f)
    mg.ir_set_guess(x0)
    res = mg.ir_solve(h, tol=1e-12, vcycles_per_iter=1, max_iter=1, raise_on_stall=False)
    x1 = mg.ir_solution()
    n0, n1 = (O.residual(x, f, flag, h)[1] for x in (x0, x1))
    assert np.abs(x1 - x0).max() > 0
    np.testing.assert_allclose([res["r0_norm"], res["rel_residual"] * res["r0_norm"]], [n0, n1],
                               rtol=6e-11)
    mg.close()


def test_batched_update_is_the_single_one(gpu):
    sizes = [s for s in SIZES if min(s) >= 16]  # the batch's smallest domain
    b = Batch(sizes)
    for d, (W, H) in enumerate(sizes):
        flag, f, x0, h = problem(W, H)
        b.set_domain(d, flag, f, h)
        b.set_guess(d, x0)
    b.solve(tol=1e-12, vcycles_per_iter=2, max_iter=2, raise_on_stall=False)
    for d, (W, H) in enumerate(sizes):
        flag, f, x0, h = problem(W, H)
        mg = U.MG(flag)
        mg.ir_set_rhs(f)
        mg.ir_set_guess(x0)
        res = mg.ir_solve(h, tol=1e-12, vcycles_per_iter=2, max_iter=2, raise_on_stall=False)
        got = b.result(d)
        assert (got["r0_norm"], got["rel_residual"]) == (res["r0_norm"], res["rel_residual"])
        np.testing.assert_array_equal(b.solution(d), mg.ir_solution(), err_msg=f"{W}x{H}")
        mg.close()
