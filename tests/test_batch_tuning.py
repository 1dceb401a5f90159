"""Entries of a tuning file that were timed with other kernels or another
relaxation factor are not taken: the batch is timed again and gets an entry of
its own, which the next autotune of the same kind takes."""
import pytest

import ubootgl_amd as U
from ubootgl_amd.batch import Batch
from ubootgl_amd import workloads as W

pytestmark = pytest.mark.gpu

SIZES = [(96, 48), (130, 70)]


def former_key(sizes, counts):
    """FNV-1a over sizes, smoothing counts and V-cycles a step, the key of a
    file written when pass_rows named the rows of LDS tiles."""
    h = 1469598103934665603
    for v in [x for s in sizes for x in s] + counts:
        for b in int(v).to_bytes(8, "little"):
            h = ((h ^ b) * 1099511628211) % 2**64
    return f"{h:016x}"


def tuned(db, alpha=1.0):
    b = Batch(SIZES, U.Params(alpha=alpha))
    for d, (w, h) in enumerate(SIZES):
        b.set_problem(d, W.poisson_problem(w, h, seed=d))
    t = b.autotune(str(db))
    b.close()
    return t


def test_entries_of_other_kernels_are_timed_again(gpu, tmp_path):
    db = tmp_path / "tune.db"
    db.write_text(former_key(SIZES, [3, 3, 5, 4]) + " 64 8 2048 32 123456\n")
    t = tuned(db)
    assert t["sweep_ms"] < 1000.0
    assert len(db.read_text().splitlines()) == 2
    # the new entry is taken: its line, marked, comes back
    lines = db.read_text().splitlines()
    f = lines[1].split()
    db.write_text("\n".join([lines[0], " ".join(f[:5] + ["4321"])]) + "\n")
    assert tuned(db)["sweep_ms"] == 4321.0
    assert tuned(db, alpha=0.8)["sweep_ms"] < 1000.0
    assert len(db.read_text().splitlines()) == 3
