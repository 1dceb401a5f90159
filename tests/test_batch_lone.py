"""A batch of one domain whose smoothing counts take a launch per sweep (its steps
are replayed from captured graphs, one per buffer state): cold and warm solves,
several on one handle with reads, eager work and another cycle count between
them, equal the single-domain solves bit for bit."""
import numpy as np
import pytest

import ubootgl_amd as U
from ubootgl_amd import workloads as W
from ubootgl_amd.batch import Batch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("w,h,pre,post", [(16, 16, 5, 5), (64, 48, 4, 1), (130, 71, 0, 20),
                                          (257, 129, 7, 4)])
def test_lone_domain_equals_single(gpu, w, h, pre, post):
    P = W.poisson_problem(w, h, seed=5, solid=0.02)
    prm = U.Params(nu_pre=pre, nu_post=post)
    b, m = Batch([(w, h)], prm), U.MG(P.flag)
    m.set_params(prm)
    b.set_problem(0, P)
    m.ir_set_rhs(P.f)
    for tol, k, cold in ((1e-8, 4, True), (1e-4, 4, True), (1e-7, 3, False), (1e-8, 4, True),
                         (1e-6, 4, True)):
        if cold:
            b.set_guess(0)
            m.ir_set_guess(None)
        b.solve(tol=tol, vcycles_per_iter=k, raise_on_stall=False)
        want = m.ir_solve(float(P.h), tol=tol, vcycles_per_iter=k, raise_on_stall=False)
        assert b.result(0) == want, (tol, k)
        np.testing.assert_array_equal(b.solution(0), m.ir_solution())
        b.set_rhs(0, P.f)
    b.close()
    m.close()
