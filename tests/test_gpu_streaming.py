"""The streaming kernels (mu-t conversion, spike removal, sinogram correction,
rotation-centre shift) at the edges of their work split: 8 rows a thread, 4
columns a thread where widths, strides and pointers are aligned and one
otherwise.  The operations of an element do not depend on the split, so results
equal the oracle's (whole-number rules, linear sampling) or, where the oracle's
libm differs by rounding, those of the other split, bit for bit."""
import numpy as np
import pytest
import torch

import oracle as O
from _util import dev, host, say

pytestmark = pytest.mark.gpu


def _off(a, skip):
    """A device copy of a that starts `skip` elements into its allocation."""
    t = torch.from_numpy(np.ascontiguousarray(a).reshape(-1).view(np.int16) if a.dtype == np.uint16
                         else np.ascontiguousarray(a).reshape(-1))
    buf = torch.zeros(t.numel() + skip, dtype=t.dtype, device="cuda")
    buf[skip:] = t.cuda()
    return buf[skip:].view(a.shape)


@pytest.mark.parametrize("skip", [0, 1])
@pytest.mark.parametrize("nz,A,W", [(1, 1, 4), (2, 7, 64), (3, 8, 66), (1, 9, 3), (5, 17, 260), (2, 16, 1025)])
def test_denoise_splits(ctx, nz, A, W, skip):
    rng = np.random.default_rng(A + W)
    src = rng.uniform(0.0, 1.0, (nz, A, W)).astype(np.float32)
    src[:, rng.integers(0, A, 20), rng.integers(0, W, 20)] += 4.0
    say("denoise", nz, A, W, skip)
    assert np.array_equal(host(ctx.denoise_sinogram(_off(src, skip), 0.8)), O.denoise_sinogram(src, 0.8))


@pytest.mark.parametrize("n,W,H,gap", [(1, 8, 1, 0), (8, 16, 33, 4), (9, 64, 20, 0), (7, 13, 11, 0), (17, 64, 9, 3)])
def test_mt_conversion_splits(ctx, n, W, H, gap):
    rng = np.random.default_rng(n + W)
    stride = W * H + gap
    dark = rng.uniform(90.0, 110.0, (H, W)).astype(np.float32)
    I0 = rng.uniform(3000.0, 4000.0, (H, W)).astype(np.float32)
    It = rng.integers(0, 5000, stride * n).astype(np.uint16)
    It[:5] = 100
    say("mt_conversion", n, W, H, gap)
    got = [host(ctx.mt_conversion(_off(dark, s), _off(I0, s), _off(It, s), n, stride)) for s in (0, 1)]
    assert np.array_equal(got[0], got[1])
    # rtol / atol: two ulp of the logarithm and of the division, as the conversion's own test
    assert np.allclose(got[0], O.mt_conversion(dark, I0, It, n, W, H, stride), rtol=2e-6, atol=2e-6)


@pytest.mark.parametrize("mode", [1, 2, 3, 4])
@pytest.mark.parametrize("nz,pa,px", [(1, 1, 8), (3, 7, 64), (2, 12, 258), (5, 9, 33)])
def test_sinogram_correction_splits(ctx, nz, pa, px, mode):
    rng = np.random.default_rng(pa + px)
    ctx.set_geometry(px, px, pa, 1, angles_deg=(np.arange(pa) * (180.0 / pa)).astype(np.float32), correction_mode=mode)
    y = rng.uniform(-1.0, 2.0, (nz, pa, px)).astype(np.float32)
    say("sinogram correction", nz, pa, px, mode)
    got = []
    for skip in (0, 1):
        out = _off(np.zeros_like(y), skip)
        ctx.op("sinogram_correction", _off(y, skip), out, nz, mode)
        ctx.synchronize()
        got.append(host(out))
    assert np.array_equal(got[0], got[1])
    for z in range(nz):                              # a row's place in its strip changes nothing
        one = dev(np.zeros((1, pa, px), np.float32))
        ctx.op("sinogram_correction", dev(y[z:z + 1]), one, 1, mode)
        ctx.synchronize()
        assert np.array_equal(host(one)[0], got[0][z]), z


@pytest.mark.parametrize("pa,px,cnt", [(1, 64, 4), (8, 33, 4), (9, 300, 5), (23, 257, 7)])
def test_rot_shift_splits(ctx, pa, px, cnt):
    ang = (np.arange(pa) * (180.0 / pa)).astype(np.float32)
    ctx.set_geometry(px, px, pa, 1, angles_deg=ang)
    prj = np.random.default_rng(pa + px).uniform(-1.0, 2.0, (pa, px)).astype(np.float32)
    say("rot shift", pa, px, cnt)
    out = dev(np.zeros((cnt, pa, px)))
    ctx.op("rot_center_shift", dev(prj), out, cnt, -2.35, 1.7)
    assert np.array_equal(host(out), O.rot_center_shift(O.geom(px, px, pa, ss=1), prj, cnt, -2.35, 1.7))
