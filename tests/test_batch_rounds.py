"""Batched solves whose member set shrinks round after round (more uploads of
tables and states than the staging has slots) and grows again with the next
solve: every domain's result and solve state equal the single-domain solve's,
bit for bit, in a cold solve, a second one on the same handle with another
tolerance, and a warm one."""
import numpy as np
import pytest

import ubootgl_amd as U
from ubootgl_amd.batch import Batch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 17, 40])
def test_rounds_match_single_solves(gpu, n):
    sizes = [(16 + 9 * i, 16 + (37 * i) % 150) for i in range(n)]
    g = np.random.default_rng(n)
    prob = []
    for W, H in sizes:
        flag = np.ones((H, W), np.float32)
        flag[2:-2, 2:-2] = g.random((H - 4, W - 4)) > 0.05
        prob.append((flag, g.standard_normal((H, W)).astype(np.float32), float(np.float32(1 / W))))
    b = Batch(sizes)
    mgs = [U.MG(p[0]) for p in prob]
    for d, (flag, f, h) in enumerate(prob):
        b.set_domain(d, flag, f, h)
        mgs[d].ir_set_rhs(f)
    for tol, cold in ((1e-9, True), (1e-5, True), (1e-2, False)):
        for d in range(n):
            if cold:
                b.set_guess(d)
                mgs[d].ir_set_guess(None)
        b.solve(tol=tol, raise_on_stall=False)
        for d, (flag, f, h) in enumerate(prob):
            want, got = mgs[d].ir_solve(h, tol=tol, raise_on_stall=False), b.result(d)
            assert got == want, (d, sizes[d], tol)
            np.testing.assert_array_equal(b.solution(d), mgs[d].ir_solution())
    for m in mgs:
        m.close()
