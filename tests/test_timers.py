"""Kernel timers of a simulation: the default one counts every level-0 launch
that smooths, whether the sweeps are launches of their own or part of a level
pass, and a launch of two classes counts for both timers."""
import numpy as np
import pytest

import ubootgl_amd as U
from ubootgl_amd import _lib as L
from ubootgl_amd import workloads as W

pytestmark = pytest.mark.gpu


def sim(nu_pre, nu_post):
    d = W.small_domain(200, 100, seed=4)
    s = U.Simulation(d.flag, d.pwidth, d.mu,
                     U.Params(nu_pre=nu_pre, nu_post=nu_post, vcycles_per_step=2))
    return s, float(d.dt)


# pre, post: smoothing counts; launches a V-cycle of the default timer: passes
# with sweeps, and the sweeps beyond a pass's three
@pytest.mark.parametrize("pre,post,launches", [(3, 3, 2), (2, 0, 1), (0, 0, 0), (5, 4, 5)])
def test_default_timer_counts_smoothing_launches(gpu, pre, post, launches):
    s, dt = sim(pre, post)
    s.step(dt)
    s.timer_enable()
    for _ in range(3):
        s.step(dt)
    ms, n = s.timer_read()
    assert n == 3 * 2 * launches
    assert ms > 0.0 if launches else ms == 0.0
    assert s.timer_read() == (ms, n)
    s.timer_enable(on=False)
    s.step(dt)
    assert s.timer_read()[1] == 0
    s.close()


def test_launch_of_two_classes_counts_for_both(gpu):
    s, dt = sim(3, 3)
    for t in (L.TIMER_L0_PRE, L.TIMER_SMOOTH_L0, L.TIMER_L0_POST, L.TIMER_ADVECT):
        s.timer_enable(t)
    for _ in range(2):
        s.step(dt)
    pre = s.timer_read(L.TIMER_L0_PRE)
    s.timer_enable(L.TIMER_L0_PRE, False)  # what it has timed stays with the other
    post = s.timer_read(L.TIMER_L0_POST)
    both = s.timer_read()
    assert pre[1] == post[1] == 4 and both[1] == 8
    np.testing.assert_allclose(both[0], pre[0] + post[0], rtol=1e-12)
    assert s.timer_read(L.TIMER_ADVECT)[1] == 2
    s.step(dt)  # the pre pass by the default timer alone
    assert s.timer_read(L.TIMER_L0_PRE) == (0.0, 0)
    assert s.timer_read()[1] == 12
    s.close()
