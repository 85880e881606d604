"""The TV-coupled OS-EM and the additive method (AART) on stacks that run as
quads (four interleaved slices), as single slices, and as both.  The kernels
keep every slice's operations and their order, so the images are equal bit for
bit to the same steps taken one public operation (TV) or one slice (AART) at a
time.  Sizes at the edges of 64-column tiles, of the four rows of a thread and
of the 16 rows of a block; whole quads, quads with empty places, slices left
over, and stacks too small for quads."""
import numpy as np
import pytest
from ctrecon import subset_order

from _util import dev, host, say

pytestmark = pytest.mark.gpu

CASES = [
    # nx, ny, px, pa, ss, dn: at least 560 filled projection and 112 backprojection blocks run as quads
    # (AART of so few subsets and blocks singly)
    (66, 53, 130, 130, 2, 58),                  # whole quads and one with two
    (64, 64, 64, 180, 2, 113),                  # whole tiles; a quad with one
    (127, 35, 65, 182, 2, 79),                  # one column short, three rows over, a quad with three
    (33, 130, 97, 90, 3, 5),                    # single slices only
    (65, 17, 40, 60, 4, 1),                     # one slice: it is its own layer neighbour
]


def _inputs(ctx, nx, ny, px, pa, ss, dn, **kw):
    rng = np.random.default_rng(nx + 3 * ny + px + dn)
    ang = (np.arange(pa) * (180.0 / pa)).astype(np.float32)
    ctx.set_geometry(nx, px, pa, ss, ny=ny, angles_deg=ang, **kw)
    x0 = rng.uniform(0.2, 1.5, (dn, ny, nx)).astype(np.float32)
    y = rng.uniform(0.0, 60.0, (dn, pa, px)).astype(np.float32)
    y[0, 0, 0] = np.nan
    return x0, y


@pytest.mark.parametrize("nx,ny,px,pa,ss,dn", CASES)
def test_tv_stack_equals_its_steps(ctx, nx, ny, px, pa, ss, dn):
    x0, y = _inputs(ctx, nx, ny, px, pa, ss, dn, cs_lambda=2e-2)
    say("tv stack", nx, ny, px, pa, ss, dn)
    it = 2
    got = dev(x0)
    ctx.fista_osem_execution(got, dev(y), it)
    x, yd, rows = dev(x0), dev(y), dev(np.zeros_like(y))
    v, w, bn, b = (dev(np.zeros_like(x0)) for _ in range(4))
    L = dev(np.full(ss, 0.5, np.float32))
    for i in range(it):
        for k, sub in enumerate(int(s) for s in subset_order(ss)):
            ctx.op("osem1", x, yd, rows, dn, sub)
            ctx.op("osem2", x, rows, v, dn, sub)
            new = dev(np.zeros_like(x0))
            if i == 0 and k == 0:
                ctx.op("ista3d", x, new, dn, sub, L)
            else:
                ctx.op("fista3d", x, v, b, w, new, bn, dn, sub, L)
            ctx.synchronize()
            x = new
    assert np.array_equal(host(got), host(x))


@pytest.mark.parametrize("nx,ny,px,pa,ss,dn", CASES)
@pytest.mark.parametrize("it", [0, 2])
def test_aart_stack_equals_single_slices(ctx, nx, ny, px, pa, ss, dn, it):
    x0, y = _inputs(ctx, nx, ny, px, pa, ss, dn, mode=2)
    say("aart stack", nx, ny, px, pa, ss, dn, it)
    got = dev(x0)
    ctx.aart_execution(got, dev(y), it)
    for z in range(dn):                          # one slice never forms a quad
        one = dev(x0[z:z + 1])
        ctx.aart_execution(one, dev(y[z:z + 1]), it)
        assert np.array_equal(host(one)[0], host(got)[z]), z
