"""Batched solves whose allocations fail (tests/cpp/batch_alloc_test.cpp, which
stands in for the HIP runtime): an error is returned, and the next call builds
its tables again instead of running over an earlier member set's."""
import os
import subprocess

CPP = os.path.join(os.path.dirname(os.path.abspath(__file__)), "cpp")


def test_failed_allocations_leave_no_stale_tables():
    out = subprocess.run(["make", "-C", CPP, "_build/batch_alloc_test"], capture_output=True,
                         text=True)
    assert out.returncode == 0, out.stdout + out.stderr
    out = subprocess.run([os.path.join(CPP, "_build", "batch_alloc_test")], capture_output=True,
                         text=True, timeout=120)
    assert out.returncode == 0, out.stdout + out.stderr
    assert "ALL OK" in out.stdout
