"""Bands and windows of the alignment forward's quads (k_align_quad), on the CPU: the
window of 2560 texels and, with the derivative, of 3328, for blocks whose two angles
have offsets of their own, from equal ones to some that take an angle off the image.
The walk and its checks are those of the projector's bounds; a ray's coordinates are
the alignment model's."""
import numpy as np
import pytest

import test_quad_bounds as tb
from test_quad_bounds import LT, QA, QEDGE, _fma, f32


class _AlignRay(tb._Ray):
    def __init__(self, nx, ny, px, c, s, ch, shift, center):
        D = max(nx, ny)
        dh = f32(D * 0.5)
        eta = (np.arange(D).astype(f32) - dh).astype(f32)
        self.tr = tr = abs(s) > abs(c)
        W, Hi = (ny, nx) if tr else (nx, ny)
        cdl, rdl = (c, s) if tr else (s, c)
        self.up = rdl > 0
        X = np.arange(ch * LT, min(ch * LT + LT - 1, px - 1) + 1)
        xi = np.clip((X.astype(f32) - f32(px * 0.5) - f32(shift)).astype(f32) - f32(center), f32(-1e30), f32(1e30)).astype(f32)
        bu, bv = _fma(xi, c, f32(nx * 0.5)), _fma(-xi, s, f32(ny * 0.5))
        cb, rb = (bv, bu) if tr else (bu, bv)
        self.slope = slope = f32(cdl / rdl)
        q = [_fma(-rb[i], slope, cb[i]) for i in (0, -1)]
        self.lo, self.hi = min(q), max(q)
        e0, e1 = f32(-dh * rdl), f32((f32(D - 1) - dh) * rdl)
        vlo = max(f32(-1) - f32(2) * QEDGE, min(rb[0], rb[-1]) + min(e0, e1) - f32(2))
        vhi = min(f32(Hi) - f32(0.5), max(rb[0], rb[-1]) + max(e0, e1) + f32(2))
        if abs(slope) < 1e-6:
            if self.lo > W + 1 or self.hi < -2:
                vhi = vlo - 1
        else:
            a, g = f32((f32(W + 1) - self.lo) / slope), f32((f32(-2) - self.hi) / slope)
            vlo, vhi = max(vlo, min(a, g) - f32(1)), min(vhi, max(a, g) + f32(1))
        self.vlo, self.vhi, self.rb, self.rdl, self.dh = vlo, vhi, rb, rdl, dh
        self.ic = np.floor(_fma(eta[None, :], cdl, cb[:, None])).astype(np.int64)
        self.ir = np.floor(_fma(eta[None, :], rdl, rb[:, None])).astype(np.int64)
        self.tap = (self.ic >= -1) & (self.ic < W) & (self.ir >= -1) & (self.ir < Hi)
        self.walked = np.zeros(self.tap.shape, bool)


@pytest.mark.parametrize("cap", [2560, 3328])
@pytest.mark.parametrize("nx,ny,px,count", [(37, 37, 41, 10), (80, 48, 64, 10), (20, 33, 400, 6), (301, 301, 256, 5),
                                            (742, 742, 512, 0), (2000, 2000, 1380, 0)])
def test_alignment_bands(monkeypatch, cap, nx, ny, px, count):
    monkeypatch.setattr(tb, "QCAP", cap)
    C, S = tb._angles(nx + 5 * ny + px, count)
    if nx >= 700:
        C, S = C[::4], S[::4]
    rng = np.random.default_rng(cap + nx)
    chunks = list(range((px + LT - 1) // LT))[::7 if nx >= 2000 else (3 if nx >= 700 else (2 if nx >= 300 else 1))]
    shared = alone = 0
    for i, (c, s) in enumerate(zip(C, S)):
        th = np.arctan2(np.float64(s), np.float64(c)) + np.deg2rad((0.1, 0.7, 3.0)[i % 3]) * np.arange(QA)
        cg, sg = np.cos(th).astype(f32), np.sin(th).astype(f32)
        cg[0], sg[0] = c, s
        near = rng.normal(0.0, 3.0, QA)
        for shift in (near, near * [1.0, 12.0], [0.25 * px, -0.5 * px], [near[0], 5000.0]):
            for ch in chunks:
                rays = [_AlignRay(nx, ny, px, cg[a], sg[a], ch, shift[a], 0.7) for a in range(QA)]
                share = tb._share(rays)
                shared, alone = shared + share, alone + (not share)
                for part in ([rays] if share else [[r] for r in rays]):
                    tb._walk(part, nx, ny)
                for r in rays:
                    assert not (r.tap & ~r.walked).any(), (float(c), float(s), ch, shift)
    assert shared > 0 and alone > 0
