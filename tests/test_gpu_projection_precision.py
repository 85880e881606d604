"""The projector's rounding on an image of noise, where the samples' fractions
decide it.  A row's distance from 64 bits is held to that of coordinates taken
relative to a tile of 60 samples (numbers below 96, a fraction of 17 bits or more),
restated here in numpy with the kernel's order of summation; fractions of numbers as
large as the image side would exceed it by 1.3 to 1.6 times.  aart1 of a zero
sinogram is the negated projection."""
import ctypes
import math

import numpy as np
import pytest

from _util import dev, host, say

f32 = np.float32


def _fma(a, b, c):
    return (np.float64(a) * np.float64(b) + np.float64(c)).astype(f32)


def _cos_sin(deg):
    libm = ctypes.CDLL("libm.so.6")
    for name in ("cosf", "sinf"):
        getattr(libm, name).restype = ctypes.c_float
        getattr(libm, name).argtypes = [ctypes.c_float]
    a = float(f32(float(f32(deg)) * math.pi / 180.0))
    return f32(libm.cosf(a)), f32(libm.sinf(a))


class _Rows:
    """Samples of the chunks' rays (64 each) of one image at one angle."""

    def __init__(self, img, deg, chunks):
        n = self.n = img.shape[0]
        c, s = _cos_sin(deg)
        self.X = np.concatenate([np.arange(64 * k, 64 * k + 64) for k in chunks])
        tr = abs(s) > abs(c)
        pad = np.zeros((n + 8, n + 8), f32)
        pad[4:-4, 4:-4] = img
        self.img = pad.T if tr else pad
        xi = (self.X.astype(f32) - f32(n * 0.5)).astype(f32)
        bu, bv = _fma(xi, c, f32(n * 0.5)), _fma(-xi, s, f32(n * 0.5))
        self.cb, self.rb = (bv, bu) if tr else (bu, bv)
        self.cdl, self.rdl = (c, s) if tr else (s, c)
        eta, xi = np.arange(n) - n * 0.5, (self.X - n * 0.5)[:, None]
        u, v = xi * np.float64(c) + n * 0.5 + eta * np.float64(s), -xi * np.float64(s) + n * 0.5 + eta * np.float64(c)
        cc, rr = (v, u) if tr else (u, v)
        self.want = self._sample(np.floor(cc).astype(int), np.floor(rr).astype(int), cc - np.floor(cc),
                                 rr - np.floor(rr)).sum(1)

    def _sample(self, ic, ir, fa, fb):
        at = lambda i: np.clip(i, -3, self.n + 2) + 4            # noqa: E731
        t = [self.img[at(ir + j), at(ic + i)] for j in (0, 1) for i in (0, 1)]
        if fa.dtype == np.float64:
            t = [x.astype(np.float64) for x in t]
            l0, l1 = t[0] + fa * (t[1] - t[0]), t[2] + fa * (t[3] - t[2])
            return l0 + fb * (l1 - l0)
        l0, l1 = _fma(fa, (t[1] - t[0]).astype(f32), t[0]), _fma(fa, (t[3] - t[2]).astype(f32), t[2])
        return _fma(fb, (l1 - l0).astype(f32), l0)

    def relative_to_tiles(self, tile=60):
        n, dh = self.n, f32(self.n * 0.5)
        vals = np.zeros((len(self.X), n), f32)
        for x0 in range(0, len(self.X), 64):
            for k0 in range(0, n, tile):
                k = np.arange(k0, min(n, k0 + tile))
                ph = (k - k0) % 4
                e0, m4 = (f32(k0) + ph.astype(f32) - dh).astype(f32)[None], (k - k0 - ph).astype(f32)[None]
                part, orgs, fr = slice(x0, x0 + 64), [], []
                for base, step in ((self.cb[part, None], self.cdl), (self.rb[part, None], self.rdl)):
                    org = int(np.floor(_fma((k.astype(f32) - dh)[None], step, base).min())) - 1
                    at = _fma(m4, step, _fma(e0, step, (base - f32(org)).astype(f32)))
                    orgs.append(np.floor(at).astype(int) + org)
                    fr.append((at - np.floor(at)).astype(f32))
                vals[part, k0:k0 + len(k)] = self._sample(orgs[0], orgs[1], fr[0], fr[1])
        ph = np.zeros((4, len(self.X)), f32)
        for k in range(n):
            ph[k % 4] += vals[:, k]
        return ph[0] + (ph[1] + ph[2] + ph[3])

    def err(self, rows):
        return np.linalg.norm(rows.astype(np.float64) - self.want) / np.linalg.norm(self.want)


@pytest.mark.gpu
@pytest.mark.parametrize("n", [320, 1024, 2048])
def test_projection_keeps_the_bits_of_its_fractions(ctx, n):
    deg = np.array([7.3, 31.0, 52.0, 83.0, 111.0, 160.0], f32)
    img = np.random.default_rng(n).uniform(0.0, 1.0, (n, n)).astype(f32)
    chunks = sorted({n // 64 // 8, n // 64 // 3, n // 64 // 2, n // 64 - 2})
    ctx.set_geometry(n, n, len(deg), 1, angles_deg=deg)
    rows = dev(np.zeros((1, len(deg), n)))
    say("projection precision", n)
    ctx.op("aart1", dev(img[None]), dev(np.zeros((1, len(deg), n))), rows, 1, 0)
    got = -host(rows)[0]
    mine, tiled = [], []
    for a, d in enumerate(deg):
        r = _Rows(img, d, chunks)
        mine.append(r.err(got[a, r.X]))
        tiled.append(r.err(r.relative_to_tiles()))
    mine, tiled = (float(np.sqrt(np.mean(np.square(e)))) for e in (mine, tiled))
    print(f"[precision] {n}^2: {mine:.3e}, relative to tiles {tiled:.3e}", flush=True)
    assert mine <= 1.1 * tiled
