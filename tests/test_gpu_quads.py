"""Stacks that run as quads (four interleaved slices) against the same stack
slice by slice.  ctr_osem_execution_noalloc always runs single slices, and a
quad's kernels sum each slice in the single-slice kernels' order with their
operations, so the images are equal bit for bit.  Sizes at the edges of
64-ray chunks and 64 x 16 pixel blocks, whole quads and quads with empty
places, detectors narrower and wider than the grid, and angle tables that are
dense, wide apart (the two angles of a block walk apart), beyond 180 degrees
and unordered."""
import numpy as np
import pytest

from _util import dev, host, say

pytestmark = pytest.mark.gpu


def _angles(kind, pa, rng):
    if kind == "dense":
        return np.arange(pa) * (180.0 / pa)
    if kind == "full":
        return np.arange(pa) * (360.0 / pa)
    if kind == "wide":
        return (np.arange(pa) * 37.0) % 180.0
    return rng.uniform(-200.0, 500.0, pa)


@pytest.mark.parametrize("nx,ny,px,pa,ss,dn,kind", [
    (128, 128, 128, 128, 1, 32, "dense"),       # whole chunks and pixel blocks
    (129, 129, 129, 130, 2, 60, "full"),        # one ray, one pixel over
    (127, 127, 127, 240, 2, 35, "random"),      # a quad with three slices
    (150, 97, 170, 105, 1, 34, "wide"),         # rectangular, wide detector, a quad with two
    (97, 150, 61, 300, 1, 33, "dense"),         # narrow detector, a quad with one
    (20, 20, 20, 64, 1, 226, "random"),         # smaller than a chunk and a block
    (512, 512, 512, 90, 1, 12, "wide"),         # angles too far apart for a window: single slices
    (1024, 1024, 1024, 240, 2, 4, "dense"),
])
def test_quads_equal_single_slices(ctx, nx, ny, px, pa, ss, dn, kind):
    rng = np.random.default_rng(nx + 3 * ny + px)
    ctx.set_geometry(nx, px, pa, ss, ny=ny, angles_deg=_angles(kind, pa, rng).astype(np.float32))
    x0 = rng.uniform(0.2, 1.5, (dn, ny, nx)).astype(np.float32)
    y = rng.uniform(0.0, 60.0, (dn, pa, px)).astype(np.float32)
    y[0, 0, 0] = np.nan
    y[dn - 1, pa // 2, px // 3] = 0.0
    say("quads", nx, ny, px, pa, ss, dn, kind)
    a = dev(x0)
    ctx.osem_execution(a, dev(y), 2)
    want = []
    for z in range(0, dn, 2):                    # pairs and single slices never form a quad
        b = dev(x0[z:z + 2])
        ctx.osem_execution_noalloc(b, dev(y[z:z + 2]), 2)
        want.append(host(b))
    assert np.array_equal(host(a), np.concatenate(want))


def test_batched_quads_equal_single_slices(ctx):
    """An uneven batched stack whose sides leave 0, 1, 2 and 3 slices past whole quads."""
    pa, ss = 120, 1
    ang = (np.arange(pa) * (180.0 / pa)).astype(np.float32)
    rng = np.random.default_rng(8)
    sides = [64] * 8 + [200] * 13 + [129] * 14 + [257] * 7 + [90] * 2 + [301]
    rng.shuffle(sides)
    ctx.set_geometry(64, 64, pa, ss, angles_deg=ang)
    x0 = [rng.uniform(0.2, 1.5, (n, n)).astype(np.float32) for n in sides]
    y = [rng.uniform(0.0, 60.0, (pa, n)).astype(np.float32) for n in sides]
    imgs, prjs = [dev(v) for v in x0], [dev(v) for v in y]
    say("batched quads", len(sides))
    ctx.osem_batched(imgs, prjs, 2, use_graph=True)
    ctx.synchronize()
    for i, n in enumerate(sides):
        ctx.set_geometry(n, n, pa, ss, angles_deg=ang)
        b = dev(x0[i][None])
        ctx.osem_execution_noalloc(b, dev(y[i][None]), 2)
        assert np.array_equal(host(b)[0], host(imgs[i])), (i, n)
