"""Every backprojection kernel of FBP on the GPU: one, two and four slices split over
waves, whole rows, and quads split and whole, the last two with empty places and
with a layer left over.  The first test holds the rows to the kernels they name, by
the library's own choice.  Layers against the oracle's FP32 restatement, to the 1e-5
of the single operators."""
import numpy as np
import pytest

import _quads
import oracle as O
from _util import dev, host, relerr, say

CASES = [
    # n, px, pa, zp, dn, layers in quads, kernels (slices side by side, rows, angle shares)
    (200, 180, 47, 512, 2, 0, {148}),            # 4 rows, 8 shares
    (512, 500, 25, 1024, 2, 0, {184}),           # 8 rows, 4 shares
    (509, 512, 7, 1024, 3, 3, {444}),            # quads of 4 rows, one empty place
    (1000, 700, 9, 2048, 1, 0, {140}),           # 16 rows
    (512, 520, 26, 2048, 5, 4, {444, 148}),      # split quads, a layer left over
    (300, 300, 41, 512, 23, 23, {440}),          # quads of 16 rows, one empty place
    (300, 300, 41, 512, 22, 22, {440}),          # two empty places
    (640, 640, 11, 2048, 9, 8, {440, 184}),
]


def test_rows_name_their_kernels():
    for n, px, pa, zp, dn, nq, kernels in CASES:
        assert _quads.fbp_kernels(n, n, zp, dn) == (nq, kernels), (n, dn)
    assert set().union(*(c[-1] for c in CASES)) == {148, 184, 140, 444, 440}


@pytest.mark.gpu
@pytest.mark.parametrize("n,px,pa,zp,dn,nq,kernels", CASES)
def test_fbp_kernels_match_oracle(ctx, n, px, pa, zp, dn, nq, kernels):
    rng = np.random.default_rng(n + px + dn)
    ang = rng.uniform(-90.0, 400.0, pa).astype(np.float32)
    y = rng.uniform(0.0, 4.0, (dn, pa, px)).astype(np.float32)
    ctx.set_geometry(n, px, pa, 1, zp=zp, angles_deg=ang)
    x = dev(np.full((dn, n, n), 7.0))
    say("fbp kernels", n, px, pa, zp, dn)
    ctx.fbp_execution(x, dev(y))
    got = host(x)
    pick = sorted({0, dn // 2, dn - 2, dn - 1} & set(range(dn)))
    want = O.fbp_execution(O.geom(n, px, pa, zp=zp), ang, y[pick])
    for k, z in enumerate(pick):
        assert relerr(got[z], want[k]) < 1e-5, z
