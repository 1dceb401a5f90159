"""The register-tiled level passes (regtile_device.hpp) at the sizes where a
tile can go wrong, bit-identical to the oracle's V-cycle: levels smaller than
a tile, widths and heights on both sides of a tile's edge, last tiles that
own a single row or column under the zero-gradient BC, odd sizes, each tile
shape of the dispatch rule, every smoothing count with a pass of its own and
one beyond, alpha off 1, and flags from all fluid to noise (uniform rows,
mixed rows, solid sides)."""
import numpy as np
import pytest

import ubootgl_amd as U
from oracle import pyoracle as O

pytestmark = pytest.mark.gpu


def flags(W, H, kind, seed):
    g = np.random.default_rng(seed)
    f = np.ones((H, W), np.float32)
    if kind == "noise":
        f[g.random((H, W)) < 0.15] = 0
    if kind == "disks":
        y, x = np.mgrid[0:H, 0:W]
        for _ in range(max(2, W * H // 4000)):
            cx, cy, r = g.uniform(0, W), g.uniform(0, H), g.uniform(2, 9)
            f[(x - cx) ** 2 + (y - cy) ** 2 <= r * r] = 0
        f[0] = f[-1] = 0
        f[:, 0] = f[:, -1] = 0
    return f


CASES = [  # W, H, smoothing, flags, alpha
    (96, 80, 3, "disks", 1.0),      # one tile column, level 0 above the LDS size
    (128, 64, 2, "open", 1.0),
    (113, 65, 3, "disks", 1.0),     # one past the pre pass's columns
    (115, 181, 3, "noise", 1.0),    # last post tile owns one row
    (6841, 24, 3, "open", 1.0),     # last post tile owns one column
    (229, 49, 1, "disks", 1.0),
    (121, 97, 0, "noise", 1.0),
    (118, 241, 2, "open", 0.8),
    (150, 90, 5, "disks", 1.0),     # more sweeps than a pass holds
    (901, 331, 3, "disks", 1.0),    # the second shape
    (1000, 421, 2, "noise", 1.0),
    (1001, 603, 3, "disks", 1.0),   # the third shape
    (1000, 602, 2, "open", 1.0),
    (2101, 1001, 3, "disks", 1.0),  # the large shape
    (2100, 1000, 2, "noise", 1.0),
]


@pytest.mark.parametrize("zg", [False, True])
@pytest.mark.parametrize("W,H,nu,kind,alpha", CASES)
def test_level_passes_bit_exact(gpu, W, H, nu, kind, alpha, zg):
    g = np.random.default_rng(W + H)
    flag = flags(W, H, kind, 7)
    f = g.standard_normal((H, W)).astype(np.float32)
    p = g.standard_normal((H, W)).astype(np.float32)
    h = float(np.float32(1.0 / W))
    mg = U.MG(flag)
    mg.set_params(U.Params(nu_pre=nu, nu_post=nu, nu_coarse=5, alpha=alpha))
    om = O.OracleMG(W, H, nu_pre=nu, nu_post=nu, alpha=alpha)
    om.update_fields(flag)
    want = p.copy()
    for _ in range(2):
        mg.solve(p, f, flag, h, zg)
        om.solve(want, f, flag, h, zg)
    np.testing.assert_array_equal(p, want)
    mg.close()


# more than 32 tiles per CU: the 12-wave shape of 6 rows, in one column of
# tiles, in two whose second owns a few columns, and in three (whole tiles of
# uniform rows in the middle)
@pytest.mark.parametrize("W,H,kind", [(20, 164101, "noise"), (115, 82107, "noise"),
                                      (300, 55013, "open")])
@pytest.mark.parametrize("zg", [False, True])
def test_largest_shape_bit_exact(gpu, W, H, kind, zg):
    test_level_passes_bit_exact(gpu, W, H, 3, kind, 1.0, zg)


# domains so elongated that the coarsest solved level is larger than the LDS
# V-cycle's usual first level (4, 6 pairs of cells per thread), beside an
# ordinary one and ones whose LDS levels have odd widths and one or two pairs
@pytest.mark.parametrize("sizes", [[(2000, 16), (200, 100)], [(2980, 17), (16, 1700)],
                                   [(75, 131), (139, 111), (33, 1000)]])
def test_batch_lds_levels_match_single(gpu, sizes):
    from ubootgl_amd.batch import Batch
    g = np.random.default_rng(3)
    b, want = Batch(sizes), []
    for d, (W, H) in enumerate(sizes):
        flag = flags(W, H, "noise", d)
        flag[0] = flag[-1] = 1
        flag[:, 0] = flag[:, -1] = 1
        # pockets without a path to the ring would be singular
        flag[1:-1, 1:-1] = np.where(g.random((H - 2, W - 2)) < 0.04, 0, 1)
        f = (g.standard_normal((H, W)) * flag).astype(np.float32)
        f[0] = f[-1] = 0
        f[:, 0] = f[:, -1] = 0
        b.set_domain(d, flag, f, 1.0 / W)
        mg = U.MG(flag)
        mg.ir_set_rhs(f)
        mg.ir_set_guess(None)
        mg.ir_solve(float(np.float32(1.0 / W)), tol=1e-5, raise_on_stall=False)
        want.append(mg.ir_solution())
        mg.close()
    b.solve(tol=1e-5, raise_on_stall=False)
    for d in range(len(sizes)):
        np.testing.assert_array_equal(b.solution(d), want[d])
    b.close()
