"""Batched V-cycles with the zero-gradient BC in every tile shape of the level
passes, bit-identical to the single-domain solve: fixed by the tuning, on domains
smaller than a tile and on ones whose last tile owns a single row or column in
the pre or the post pass, and chosen by the members' tiles together."""
import numpy as np
import pytest

import ubootgl_amd as U
from ubootgl_amd.batch import Batch

pytestmark = pytest.mark.gpu


def domain(W, H, seed):
    g = np.random.default_rng(seed)
    flag = np.ones((H, W), np.float32)
    if seed % 3:  # every third domain is open (uniform rows, no walls)
        flag[g.random((H, W)) < 0.1] = 0
        flag[0] = flag[-1] = 0
        flag[:, 0] = flag[:, -1] = 0
    f, p = g.standard_normal((2, H, W)).astype(np.float32)
    return flag, f, p, float(np.float32(1.0 / W))


def check(sizes, nu, rows, zg=True):
    prm = U.Params(nu_pre=nu, nu_post=nu)
    b = Batch(sizes, prm)
    doms = [domain(W, H, i) for i, (W, H) in enumerate(sizes)]
    for i, (flag, f, p, h) in enumerate(doms):
        b.set_projection_domain(i, flag, f, h)
        b.set_pressure(i, p)
    b.set_tuning(64, 8, 0, rows)
    b.vcycles(2, zg)
    for i, (flag, f, p, h) in enumerate(doms):
        m = U.MG(flag)
        m.set_params(prm)
        want = p.copy()
        for _ in range(2):
            m.solve(want, f, flag, h, zg)
        m.close()
        np.testing.assert_array_equal(b.pressure(i), want, err_msg=f"domain {i} {sizes[i]}")
    b.close()


# one column left for the last tile at 1, 2 and 3 sweeps (both passes), and
# heights that leave one row: of 16-row and 32-row regions, of 48-row ones
WIDTH = {1: 7321, 2: 6845, 3: 6385}
HEIGHTS = {(1, 32): (217, 225), (2, 32): (221, 217), (3, 32): (209, 221),
           (1, 48): (201, 221), (2, 48): (217, 201), (3, 48): (225, 217)}


@pytest.mark.parametrize("rows", [8, 16, 32])
@pytest.mark.parametrize("nu", [1, 2, 3])
def test_fixed_shapes(gpu, nu, rows):
    hp, hq = HEIGHTS[nu, 48 if rows == 32 else 32]
    check([(WIDTH[nu], hp), (WIDTH[nu], hq), (16, 16), (37, 23), (64, 200), (257, 129), (130, hp),
           (201, hq)], nu, rows)


# 500x300: at most 85 tiles of the two small shapes in a pass, so 1, 3, 8 and
# 24 of them take the four shapes
@pytest.mark.parametrize("n", [1, 3, 8, 24])
@pytest.mark.parametrize("nu", [2, 3])
def test_shapes_by_tiles(gpu, nu, n):
    check([(500, 300)] * n + [(97, 61)], nu, 0)
