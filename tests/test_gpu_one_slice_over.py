"""Stacks that leave one slice over whole quads: up to a side the slice joins as a
quad with empty places, beyond it the slice runs by itself after the quads, and where
neither pays all run singly.  The kernel timing counts the parts (one projection
launch each per subset), for the drivers and for a batch of the same slices, and the
images are those of the slices run one by one, bit for bit."""
import numpy as np
import pytest

import _quads
from _util import dev, host, say

pytestmark = pytest.mark.gpu

CASES = [
    # n, px, na, dn, layers run as quads
    (256, 256, 60, 21, 0),                       # 630 blocks with a quad more: all singly
    (256, 256, 94, 13, 0),
    (256, 256, 160, 13, 13),                     # a quad more
    (512, 448, 116, 9, 9),                       # the largest side of that, just above its line
    (512, 448, 114, 9, 0),                       # just below
    (513, 513, 144, 5, 4),                       # the slice by itself, just above its line
    (520, 512, 158, 5, 0),                       # just below
    (512, 512, 172, 9, 8),                       # as little work as it does not join with
    (768, 768, 100, 5, 0),
    (128, 128, 240, 5, 0),
]


def _angles(pa):
    return (np.arange(pa) * (180.0 / pa)).astype(np.float32)


def _launches(ctx, call):
    ctx.set_kernel_timing(True)
    try:
        call()
        ctx.synchronize()
        return ctx.kernel_timing()[2]
    finally:
        ctx.set_kernel_timing(False)


@pytest.mark.parametrize("n,px,na,dn,nq", CASES)
def test_one_slice_over(ctx, n, px, na, dn, nq):
    ang = _angles(na)
    assert _quads.stack_quads(n, n, px, na, 1, dn, ang) == nq
    ctx.set_geometry(n, px, na, 1, angles_deg=ang)
    rng = np.random.default_rng(n + dn)
    x0 = rng.uniform(0.2, 1.5, (dn, n, n)).astype(np.float32)
    y = dev(rng.uniform(0.0, 60.0, (dn, na, px)).astype(np.float32))
    parts = (nq > 0) + (nq < dn)
    say("one slice over", n, px, na, dn)
    x = dev(x0)
    assert _launches(ctx, lambda: ctx.osem_execution(x, y, 1)) == parts
    got = host(x)
    for z in (0, dn - 2, dn - 1):
        one = dev(x0[z:z + 1])
        ctx.osem_execution(one, y[z:z + 1].contiguous(), 1)
        assert np.array_equal(host(one)[0], got[z]), z
    for it in (1, 8):                           # AART of few subsets needs more blocks
        nqa = _quads.stack_quads(n, n, px, na, 1, dn, ang, passes=it)
        xa = dev(x0)
        assert _launches(ctx, lambda: ctx.aart_execution(xa, y.clone(), it)) == it * ((nqa > 0) + (nqa < dn))
        for z in (0, dn - 1):
            one = dev(x0[z:z + 1])
            ctx.aart_execution(one, y[z:z + 1].clone(), it)
            assert np.array_equal(host(one)[0], host(xa)[z]), (it, z)
    assert nqa == nq
    if px == n:                                  # a batch's detector is its side
        imgs = [dev(v) for v in x0]
        assert _launches(ctx, lambda: ctx.osem_batched(imgs, [y[z] for z in range(dn)], 1, use_graph=False)) == parts
        assert all(np.array_equal(host(im), got[z]) for z, im in enumerate(imgs))


@pytest.mark.parametrize("n,px,pa,dn,nq", [
    (128, 128, 900, 5, 0), (130, 65, 903, 9, 9), (520, 512, 400, 5, 4), (256, 256, 340, 9, 9), (256, 256, 200, 9, 0),
    (256, 256, 700, 9, 8), (33, 400, 900, 4, 4)])
@pytest.mark.parametrize("deriv", [False, True])
def test_one_layer_over_in_the_alignment_forward(ctx, n, px, pa, dn, nq, deriv):
    """Equal to one layer at a time, with offsets, and NaN for an angle whose offset is
    NaN, in the quads and in the layer left over alike."""
    ang = (np.arange(pa) * (360.0 / pa) + 0.37).astype(np.float32)
    assert _quads.align_quads(n, n, px, pa, dn, ang) == nq
    ctx.set_geometry(n, px, pa, 1, angles_deg=ang)
    rng = np.random.default_rng(n + dn)
    sh = rng.normal(0.0, 2.0, pa).astype(np.float32)
    sh[pa // 3] = np.nan
    x, shifts = dev(rng.uniform(-0.5, 1.0, (dn, n, n)).astype(np.float32)), dev(sh)
    say("one layer over", n, px, pa, dn, deriv)

    def forward(img):
        p, d = (dev(np.full((img.shape[0], pa, px), 7.0, np.float32)) for _ in range(2))
        if deriv:
            ctx.align_forward_deriv(img, shifts, 0.7, p, d)
        else:
            ctx.align_forward(img, shifts, 0.7, p)
        ctx.synchronize()
        return host(p), host(d)

    got = forward(x)
    for z in (0, dn - 2, dn - 1):
        one = forward(x[z:z + 1].contiguous())
        for k in range(2):
            assert np.array_equal(got[k][z], one[k][0], equal_nan=True), z
    for k in range(2 if deriv else 1):
        assert np.isnan(got[k][:, pa // 3]).all() and np.isfinite(np.delete(got[k], pa // 3, axis=1)).all()
