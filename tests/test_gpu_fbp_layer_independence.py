"""FBP layers of a stack do not touch each other: a layer keeps its image bit for
bit when the layers beside it hold a NaN, an infinity, or values of a very
different scale.  The stacks run as interleaved quads (512 blocks of 64 x 4 pixels
or more), whole, with an empty place, and with a layer left over; an even and an
odd number of angles (the last one has no partner in the filter's transform)."""
import numpy as np
import pytest

from _util import dev, host, say

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,px,pa,zp,dn", [
    (256, 256, 24, 512, 8), (256, 230, 25, 512, 7), (300, 333, 13, 1024, 9), (1000, 1030, 7, 4096, 4),
])
@pytest.mark.parametrize("bad", [np.nan, np.inf, 3.0e7])
def test_fbp_layers_are_independent(ctx, n, px, pa, zp, dn, bad):
    rng = np.random.default_rng(n + px + dn)
    ang = rng.uniform(0.0, 180.0, pa).astype(np.float32)
    y = rng.uniform(0.0, 4.0, (dn, pa, px)).astype(np.float32)
    ctx.set_geometry(n, px, pa, 1, zp=zp, angles_deg=ang)
    say("fbp layers", n, px, pa, zp, dn, bad)

    def run(sino):
        x = dev(np.zeros((dn, n, n)))
        ctx.fbp_execution(x, dev(sino))
        return host(x)

    want = run(y)
    for z in (0, dn // 2, dn - 1):
        spoilt = y.copy()
        if np.isfinite(bad):
            spoilt[z] *= bad
        else:
            spoilt[z, pa // 2, px // 3] = bad
        got = run(spoilt)
        rest = np.arange(dn) != z
        assert np.array_equal(got[rest], want[rest]), z
        assert not np.array_equal(got[z], want[z])
