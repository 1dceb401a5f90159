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
    (1001, 603, 3, "disks", 1.0),   # the middle shape
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
