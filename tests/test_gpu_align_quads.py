"""The alignment forward (alone and with its derivative) on stacks that run as
quads, against the same stack one layer at a time (one layer never forms a
quad).  A quad takes every layer's samples and sums in the single-layer
kernel's order, so the rows are equal bit for bit.  Sizes at the edges of
64-ray chunks, an odd number of angles, quads with empty places and layers left
over, wide and narrow detectors, offsets that differ from angle to angle, that
take an angle off the image or that are NaN."""
import numpy as np
import pytest

from _util import dev, host, say

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx,ny,px,pa,dn,spread", [
    (64, 64, 64, 1800, 4, 1.5),                 # one chunk, one quad
    (97, 61, 130, 601, 6, 12.0),                # odd angles, one column over, a quad with two
    (130, 171, 65, 903, 9, 0.0),                # one ray over, a quad with one
    (301, 301, 256, 151, 11, 90.0),             # a quad with three, angles far apart in offset
    (20, 33, 400, 257, 4, 5.0),                 # a detector much wider than the image: single layers
])
@pytest.mark.parametrize("deriv", [False, True])
def test_quads_equal_single_layers(ctx, nx, ny, px, pa, dn, spread, deriv):
    rng = np.random.default_rng(nx + 3 * ny + px)
    ang = (np.arange(pa) * (360.0 / pa) + 0.37).astype(np.float32)
    ang[::7] = rng.choice([0.0, 45.0, 90.0, 135.0, 180.0, -90.0], ang[::7].size)
    ctx.set_geometry(nx, px, pa, 1, ny=ny, angles_deg=ang)
    shifts = (spread * rng.normal(0.0, 1.0, pa)).astype(np.float32)
    shifts[::11] = rng.choice([-5000.0, 5000.0, 0.25 * px, -0.5 * px], shifts[::11].size)
    x = dev(rng.uniform(-0.5, 1.0, (dn, ny, nx)).astype(np.float32))
    say("align quads", nx, ny, px, pa, dn, spread, deriv)

    def forward(img, sh):
        p, d = (dev(np.full((img.shape[0], pa, px), 7.0, np.float32)) for _ in range(2))
        if deriv:
            ctx.align_forward_deriv(img, sh, 0.7, p, d)
        else:
            ctx.align_forward(img, sh, 0.7, p)
        ctx.synchronize()
        return host(p), host(d)

    for sh in (dev(shifts), None):
        got = forward(x, sh)
        for z in range(dn):
            one = forward(x[z:z + 1].contiguous(), sh)
            assert np.array_equal(got[0][z], one[0][0]), z
            assert np.array_equal(got[1][z], one[1][0]), z
    # NaN offsets: the stacks whose layers are all in quads
    if dn % 4 == 1:
        return
    bad = shifts.copy()
    bad[pa // 2] = np.nan
    nan = forward(x, dev(bad))
    got = forward(x, dev(shifts))
    rest = np.arange(pa) != pa // 2
    for k in range(2 if deriv else 1):
        assert np.isnan(nan[k][:, pa // 2]).all()
        assert np.array_equal(nan[k][:, rest], got[k][:, rest])
