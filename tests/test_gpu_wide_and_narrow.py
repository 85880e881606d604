"""Detectors much wider than the image and images much longer than wide: most
projection blocks have no or little work there, and stacks run slice by slice where
the rest would not fill quads.  Launches per subset tell the parts, images are those
of single slices bit for bit.  FBP of tall images counts the rows of its disk."""
import numpy as np
import pytest

import _quads
import oracle as O
from _util import dev, host, relerr, say


def _angles(pa):
    return (np.arange(pa) * (180.0 / pa)).astype(np.float32)


@pytest.mark.gpu
@pytest.mark.parametrize("nx,ny,px,na,dn,nq", [
    (520, 520, 2080, 48, 5, 0), (1024, 64, 1024, 60, 9, 0), (64, 1024, 1024, 60, 9, 0),
    (520, 520, 2080, 160, 5, 4),                 # wide, with work enough for a quad
    (700, 520, 700, 130, 5, 4),
])
def test_empty_blocks_make_no_quads(ctx, nx, ny, px, na, dn, nq):
    ang = _angles(na)
    assert _quads.stack_quads(nx, ny, px, na, 1, dn, ang) == nq
    ctx.set_geometry(nx, px, na, 1, ny=ny, angles_deg=ang)
    rng = np.random.default_rng(nx + px)
    x0 = rng.uniform(0.2, 1.5, (dn, ny, nx)).astype(np.float32)
    y = dev(rng.uniform(0.0, 60.0, (dn, na, px)).astype(np.float32))
    x = dev(x0)
    say("empty blocks", nx, ny, px, na, dn)
    ctx.set_kernel_timing(True)
    try:
        ctx.osem_execution(x, y, 1)
        ctx.synchronize()
        launches = ctx.kernel_timing()[2]
    finally:
        ctx.set_kernel_timing(False)
    assert launches == (nq > 0) + (nq < dn)
    for z in (0, dn - 1):
        one = dev(x0[z:z + 1])
        ctx.osem_execution(one, y[z:z + 1].contiguous(), 1)
        assert np.array_equal(host(one)[0], host(x)[z]), z


def test_alignment_forward_counts_the_same():
    ang = _angles(120)
    assert _quads.align_quads(198, 198, 792, 60, 12, ang[::2]) == 0
    assert _quads.align_quads(1197, 116, 1197, 120, 4, ang) == 0
    assert _quads.align_quads(241, 34, 111, 812, 8, _angles(812)) == 8
    assert _quads.align_quads(398, 398, 398, 243, 6, _angles(243)) == 0
    assert _quads.align_quads(398, 398, 398, 243, 8, _angles(243)) == 8
    assert _quads.align_quads(256, 256, 2048, 100, 4, _angles(100)) == 0
    assert _quads.align_quads(284, 284, 738, 1123, 9, _angles(1123)) == 0
    assert _quads.align_quads(284, 284, 430, 1123, 9, _angles(1123)) == 8
    assert _quads.align_quads(533, 533, 533, 240, 4, ang) == 4


def test_fbp_counts_the_rows_of_its_disk():
    assert _quads.fbp_kernels(64, 2048, 128, 16) == (0, {148})
    assert _quads.fbp_kernels(2048, 64, 4096, 16)[0] == 16


@pytest.mark.gpu
@pytest.mark.parametrize("nx,ny,px,pa,zp,dn", [(64, 2048, 64, 40, 128, 16), (130, 900, 200, 31, 512, 9),
                                               (900, 70, 333, 24, 1024, 8)])
def test_fbp_of_long_images(ctx, nx, ny, px, pa, zp, dn):
    rng = np.random.default_rng(nx)
    ang = rng.uniform(0.0, 180.0, pa).astype(np.float32)
    y = rng.uniform(0.0, 4.0, (dn, pa, px)).astype(np.float32)
    ctx.set_geometry(nx, px, pa, 1, ny=ny, zp=zp, angles_deg=ang)
    x = dev(np.full((dn, ny, nx), 7.0))
    say("fbp of long images", nx, ny, px, pa, dn)
    ctx.fbp_execution(x, dev(y))
    got = host(x)
    for z in (0, dn - 1):
        want = O.fbp_execution(O.geom(nx, px, pa, ny=ny, zp=zp), ang, y[z:z + 1])
        assert relerr(got[z], want[0]) < 1e-5, z
