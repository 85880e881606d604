"""FBP over shapes its backprojection chooses kernels by: 4 rows split over waves,
16 rows per block, and interleaved quads of layers (whole, and with one
or two empty places), on zero-padding lengths that are powers of 4 and twice
them, odd grids and detectors narrower and wider than the grid.  Every layer
against the oracle's FP32 restatement, to the 1e-5 of the single operators."""
import numpy as np
import pytest

import oracle as O
from _util import dev, host, relerr, say

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,px,pa,zp,dn", [
    (2, 2, 3, 2, 1), (3, 3, 5, 4, 2), (8, 8, 5, 8, 1), (20, 17, 7, 32, 5),
    (129, 100, 23, 128, 3),       # 4 split rows per block, an odd angle count
    (300, 390, 41, 512, 3),       # the same, a wide detector
    (257, 257, 24, 1024, 20),     # whole quads of 16 rows per block, a pixel over
    (300, 260, 40, 512, 35),      # quads of 16 rows per block, the last with three layers
    (300, 260, 39, 512, 34),      # ... with two
    (300, 300, 25, 512, 33),      # ... and one layer singly
    (1000, 1030, 25, 2048, 1),    # 16 rows per block
    (260, 250, 26, 8192, 20),     # no quads: the padding is too long for two transforms in a block
])
def test_fbp_stack_matches_oracle(ctx, n, px, pa, zp, dn):
    rng = np.random.default_rng(n + px + dn)
    ang = rng.uniform(-90.0, 400.0, pa).astype(np.float32)
    y = rng.uniform(0.0, 4.0, (dn, pa, px)).astype(np.float32)
    ctx.set_geometry(n, px, pa, 1, zp=zp, angles_deg=ang)
    x = dev(np.full((dn, n, n), 7.0))
    say("fbp stack", n, px, pa, zp, dn)
    ctx.fbp_execution(x, dev(y))
    got = host(x)
    pick = sorted({0, dn // 2, dn - 2, dn - 1} & set(range(dn)))
    want = O.fbp_execution(O.geom(n, px, pa, zp=zp), ang, y[pick])
    for k, z in enumerate(pick):
        assert relerr(got[z], want[k]) < 1e-5, z
