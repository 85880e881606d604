"""The alignment adjoint against FP64 at sizes where its two loops meet: tiles
whose pixels all lie within D/2 - 2 of the centre (no step of a window outside
[0, D)) and tiles that reach past it; even and odd D, wide and tall images,
tiles cut by the edge, and angle counts on either side of a chunk (8, 16 and 64
angles for 16, 4 and 1 slices staged together)."""
import numpy as np
import pytest

import oracle as O
from _util import dev, host, relerr, say

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx,ny,px,pa,dn", [
    (36, 36, 60, 65, 1),                        # the inner tile touches D/2 - 2
    (33, 47, 80, 64, 1),                        # odd D, a tall image: every column inside
    (130, 20, 150, 17, 3),                      # a wide image
    (49, 49, 40, 9, 5),                         # a detector narrower than the image
    (64, 64, 96, 16, 17),                       # fives of four slices, the last with one
    (272, 260, 40, 17, 17),                     # a chunk of sixteen slices and one of one
])
def test_adjoint_windows(ctx, nx, ny, px, pa, dn):
    rng = np.random.default_rng(nx + 3 * ny + dn)
    ang = (np.arange(pa) * (360.0 / pa) + 0.37).astype(np.float32)
    ang[:4] = [0.0, 45.0, 90.0, -135.0][:min(4, pa)]
    ctx.set_geometry(nx, px, pa, 1, ny=ny, angles_deg=ang)
    g = O.geom(nx, px, pa, ss=1, ny=ny)
    shifts = rng.normal(0.0, 1.5, pa).astype(np.float32)
    y = rng.normal(0.0, 1.0, (dn, pa, px)).astype(np.float32)
    say("adjoint windows", nx, ny, px, pa, dn)
    out = dev(np.zeros((dn, ny, nx)))
    ctx.align_adjoint(dev(y), dev(shifts), 0.4, out)
    exp = O.align_adjoint(g, ang, y, shifts, 0.4)
    # the bound of the FP32 oracle: coordinates rounded to FP32 near the image's side
    bound = max(1e-5, 2.0 * relerr(O.align_adjoint(g, ang, y, shifts, 0.4, dtype=np.float32), exp))
    assert relerr(host(out), exp) <= bound
