"""A served request that ends with its first update, then one on another
geometry: the step takes its own member's tables, also where the new domain sits
at the released one's address (tests/cpp/serve_members_test.cpp on the CPU; on
the GPU the answers)."""
import os
import subprocess

import numpy as np
import pytest

import ubootgl_amd as U
from ubootgl_amd import workloads as W
from ubootgl_amd.serve import Server

CPP = os.path.join(os.path.dirname(os.path.abspath(__file__)), "cpp")


def test_every_step_uploads_its_members():
    out = subprocess.run(["make", "-C", CPP, "_build/serve_members_test"], capture_output=True,
                         text=True)
    assert out.returncode == 0, out.stdout + out.stderr
    out = subprocess.run([os.path.join(CPP, "_build", "serve_members_test")], capture_output=True,
                         text=True, timeout=120)
    assert out.returncode == 0, out.stdout + out.stderr
    assert "ALL OK" in out.stdout


@pytest.mark.gpu
def test_request_after_one_without_steps(gpu):
    probs = [W.poisson_problem(w, h, seed=i) for i, (w, h) in enumerate([(96, 48), (130, 70)])]
    s = Server(hbm_budget=10**8, tol=1e-6)
    gid = [s.add_geometry(P.flag, P.h) for P in probs]
    for k in range(4):
        Z, P = probs[k % 2], probs[1 - k % 2]
        r = s.wait(s.submit(gid[k % 2], [np.zeros_like(Z.f)], want_x=True))
        assert r["iterations"] == 0 and not r["x"].any()
        r = s.wait(s.submit(gid[1 - k % 2], [P.f], want_x=True))
        m = U.MG(P.flag)
        m.ir_set_rhs(P.f)
        want = m.ir_solve(float(P.h), tol=1e-6)
        assert r["converged"] and r["iterations"] == want["iterations"]
        np.testing.assert_array_equal(r["x"], m.ir_solution())
        m.close()
    s.close()
