"""Bounds of the projector and backprojector of quads (four interleaved slices
of one geometry), checked on the CPU.

The projector (k_fp_quad) walks a block's 64 rays at two consecutive angles by
bands of image rows and stages each band's window of at most QCAP texels from
a frame QPAD texels wide.  This restates its band heights and range, windows
and sample order in float32 numpy and checks that a loaded window fits its LDS pitch and lies in
the frame, that both taps of both rows of every sample of a band lie in the
band's window, and that every sample with a tap in the image lies in a band
that is walked.

The backprojector (k_bp_quad) stages segments of 68 bins for blocks of 64 x 16
pixels; the bin rule is the single-slice kernel's.
"""
import numpy as np
import pytest

from ctrecon._lib import query_layout

f32 = np.float32
LT, QPAD, QEDGE = 64, 96, f32(0.01)
QA, QCAP, QBW = 2, 2560, 180     # angles of a block, texels and widest columns of its window
QHT_MIN, QHT_MAX = 8, 48         # rows of a band
QBP_ROWS, QBP_SEG = 4, 68


def _fma(a, b, c):
    return (np.asarray(a, np.float64) * np.asarray(b, np.float64) + np.asarray(c, np.float64)).astype(f32)


def _angles(seed, count):
    rng = np.random.default_rng(seed)
    deg = np.concatenate([np.array([0.0, 1e-4, 0.01, 44.99, 45.0, 45.01, 89.999, 90.0, 134.99, 135.0, 179.99, 180.0, 225.0,
                                    270.0, 315.0, 300.0]), rng.uniform(0.0, 360.0, count)])
    ap = (deg.astype(f32).astype(np.float64) * np.pi / 180.0).astype(f32)
    return np.cos(ap).astype(f32), np.sin(ap).astype(f32)


class _Ray:
    """The strip and samples of one 64-ray chunk at one angle."""

    def __init__(self, nx, ny, px, c, s, ch, power):
        D = max(nx, ny)
        if power:
            xh, dh = f32(px // 2), f32(D // 2)
            cu, cv = f32(f32(nx // 2) - f32(0.5)), f32(f32(ny // 2) - f32(0.5))
        else:
            xh, dh = f32(px * 0.5), f32(D * 0.5)
            cu, cv = f32(nx * 0.5), f32(ny * 0.5)
        eta = (np.arange(D).astype(f32) - dh).astype(f32)
        self.tr = tr = abs(s) > abs(c)
        W, Hi = (ny, nx) if tr else (nx, ny)
        cdl, rdl = (c, s) if tr else (s, c)
        self.up = rdl > 0
        X0, Xl = ch * LT, min(ch * LT + LT - 1, px - 1)
        X = np.arange(X0, Xl + 1)
        xi = (X.astype(f32) - xh).astype(f32)
        bu, bv = _fma(xi, c, cu), _fma(-xi, s, cv)
        cb, rb = (bv, bu) if tr else (bu, bv)
        slope = f32(cdl / rdl)
        q = [_fma(-rb[i], slope, cb[i]) for i in (0, -1)]
        self.lo, self.hi, self.slope = min(q), max(q), slope
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
        assert (np.diff(self.ir, axis=1) * (1 if self.up else -1) >= 0).all()       # rows are monotone in k
        self.tap = (self.ic >= -1) & (self.ic < W) & (self.ir >= -1) & (self.ir < Hi)
        self.walked = np.zeros(self.tap.shape, bool)


def _span(rays):
    """The rows walked, the width of the strips' union over them and the
    columns it gains per row of a band."""
    live = [r for r in rays if r.vlo <= r.vhi]
    if not live:
        return None
    v0, v1 = min(r.vlo for r in live), max(r.vhi for r in live)
    ms = f32(max([f32(0)] + [r.slope for r in rays]) - min([f32(0)] + [r.slope for r in rays]))
    ends = (f32(v0 - QHT_MAX), f32(v1 + QHT_MAX))
    w = max(max(_fma(v, r.slope, r.hi) for r in rays) - min(_fma(v, r.slope, r.lo) for r in rays) for v in ends)
    return v0, v1, f32(w), ms


def _height(w, ms):
    q = f32(w + f32(14))
    r, k = _fma(f32(2), ms, q), f32(QCAP - f32(2) * q)
    return min(QHT_MAX, int(f32(2) * k / (r + np.sqrt(max(f32(0), _fma(r, r, f32(4) * ms * k))))))


def _share(rays):
    if any(r.tr != rays[0].tr or r.up != rays[0].up for r in rays):
        return False
    sp = _span(rays)
    if sp is None:
        return True
    h = _height(sp[2], sp[3])
    return h >= QHT_MIN and sp[2] + sp[3] * f32(h) + 6 <= QBW


def _walk(rays, nx, ny):
    sp = _span(rays)
    if sp is None:
        return
    v0, v1, w, ms = sp
    tr, up = rays[0].tr, rays[0].up
    W, Hi = (ny, nx) if tr else (nx, ny)
    pitch = (W + 2 * QPAD + 15) // 16 * 16
    D = max(nx, ny)
    HT = _height(w, ms)
    bw = int(w + ms * f32(HT)) + 6
    lw = bw + ((4 - bw) & 7)
    assert HT >= QHT_MIN and bw <= QBW and lw % 8 == 4 and bw <= lw and lw * (HT + 2) <= QCAP, (HT, bw, lw)
    d0, d1 = (v0 + 2, v1 + 2) if up else (Hi - v1, Hi - v0)
    iht = f32(1) / f32(HT)
    b0, b1 = max(0, int(f32(d0) * iht)), int(f32(d1) * iht)
    ph, k = np.arange(4), np.arange(D)
    mmax = (D - ph + 3) // 4

    def upto(r, R):
        qm = f32(f32(0.25) / r.rdl)
        wm = _fma(-r.rb[:, None], qm, (f32(0.25) * (r.dh - ph.astype(f32))).astype(f32)[None, :])
        return np.clip(np.ceil(_fma(f32(f32(R) + QEDGE), qm, wm)), 0, mmax[None, :]).astype(np.int64)

    ms_ = [upto(r, -2 + b0 * HT if up else Hi - b0 * HT) for r in rays]
    for b in range(b0, b1 + 1):
        R0 = -2 + b * HT if up else Hi - (b + 1) * HT
        bx0 = int(np.floor(min(_fma(f32(R0), r.slope, f32(r.lo + min(f32(0), f32(HT) * r.slope) - f32(1))) for r in rays)))
        for a, r in enumerate(rays):
            m, mE = ms_[a], upto(r, R0 + HT if up else R0)
            ms_[a] = mE
            assert (mE >= m).all()
            nmin = int(f32(HT) * abs(f32(f32(0.25) / r.rdl)) - f32(0.002))
            full = (m > 0) & (mE < mmax[None, :])
            assert (mE - m)[full].min(initial=nmin) >= nmin and (mE - m).max(initial=0) <= nmin + 2
            inb = (k[None, :] // 4 >= m[:, k % 4]) & (k[None, :] // 4 < mE[:, k % 4])
            if bx0 >= W or bx0 + bw <= 0:
                assert not (r.tap & inb).any()
                continue
            if inb.any():
                assert r.ic[inb].min() >= bx0 and r.ic[inb].max() + 1 < bx0 + bw
                assert r.ir[inb].min() >= R0 and r.ir[inb].max() <= R0 + HT
            assert not (r.walked & inb).any()          # each sample once
            r.walked |= inb
        if not (bx0 >= W or bx0 + bw <= 0):
            # the window, rows R0 .. R0 + HT + 1 and columns bx0 .. bx0 + bw - 1, lies in the
            # frame's rows; past the frame's columns it meets the next row's zeros
            assert R0 + QPAD >= 1 and R0 + HT + 1 + QPAD < Hi + 2 * QPAD - 1
            assert bx0 >= -QPAD - QPAD and bx0 + bw <= W + QPAD + QPAD


@pytest.mark.parametrize("nx,ny,px,count", [(2, 2, 2, 14), (37, 37, 41, 14), (80, 48, 64, 14), (100, 7, 3, 14),
                                            (7, 100, 130, 14), (255, 255, 255, 8), (256, 256, 384, 6),
                                            (515, 515, 515, 4), (1024, 1024, 1024, 0), (3840, 3840, 3840, 0),
                                            (3840, 64, 3840, 0)])
@pytest.mark.parametrize("power", [False, True])
def test_projector_bands(nx, ny, px, count, power):
    if max(nx, ny) >= 1024 and power:
        pytest.skip("the other geometry rule differs by half a texel")
    C, S = _angles(nx + 5 * ny + px, count)
    if nx >= 1024:
        C, S = C[::2], S[::2]
    chunks = list(range((px + LT - 1) // LT))[::7 if px >= 3840 else (2 if px >= 1024 else 1)]
    shared = alone = 0
    for i, (c, s) in enumerate(zip(C, S)):
        th = np.arctan2(np.float64(s), np.float64(c)) + np.deg2rad((0.3, 1.5, 4.0)[i % 3]) * np.arange(QA)
        cg, sg = np.cos(th).astype(f32), np.sin(th).astype(f32)
        cg[0], sg[0] = c, s
        for ch in chunks:
            rays = [_Ray(nx, ny, px, cg[a], sg[a], ch, power) for a in range(QA)]
            share = _share(rays)
            shared, alone = shared + share, alone + (not share)
            for part in ([rays] if share else [[r] for r in rays]):
                _walk(part, nx, ny)
            for r in rays:
                assert not (r.tap & ~r.walked).any(), (float(c), float(s), ch)
    assert shared > 0 and alone > 0


@pytest.mark.parametrize("nx,ny,px", [(1024, 1024, 1024), (37, 37, 41), (80, 48, 64), (2048, 2048, 2048)])
def test_backprojector_segments(nx, ny, px):
    l = query_layout(nx, ny, px)
    rng = np.random.default_rng(nx + ny)
    C, S = _angles(nx, 60)
    C, S = C[:, None, None], S[:, None, None]
    rows = 4 * QBP_ROWS
    tiles = [(tx, ty) for tx in range((nx + 63) // 64) for ty in range((ny + rows - 1) // rows)]
    if len(tiles) > 14:
        tiles = [tiles[0], tiles[-1]] + [tiles[i] for i in rng.choice(len(tiles), 12, replace=False)]
    for tx, ty in tiles:
        X = np.minimum(tx * 64 + np.arange(64), nx - 1)
        Y = np.minimum(ty * rows + np.arange(rows), ny - 1)
        for int_half in (False, True):
            hx, hy, hp = (f32(nx // 2), f32(ny // 2), f32(px // 2)) if int_half else \
                (f32(nx * 0.5), f32(ny * 0.5), f32(px * 0.5))
            xr, yr = (X.astype(f32) - hx)[None, None, :], (Y.astype(f32) - hy)[None, :, None]
            bx = (((xr * C).astype(f32) - (yr * S).astype(f32)).astype(f32) + hp).astype(f32)
            for add_half in (False, True):
                b = np.floor(bx.astype(np.float64) + (0.5 if add_half else 0.0))
                lo = np.min(b[:, [0, 0, -1, -1], [0, -1, 0, -1]], axis=1)
                hi = np.max(b[:, [0, 0, -1, -1], [0, -1, 0, -1]], axis=1)
                assert (b >= lo[:, None, None]).all() and (b <= hi[:, None, None]).all()
                assert (hi - lo + 1).max() <= QBP_SEG
                assert lo.min() + l.roff >= 0 and hi.max() + l.roff < l.rpitch


@pytest.mark.parametrize("rows,seg", [(4, 72), (8, 72), (16, 72)])
@pytest.mark.parametrize("n,px", [(1024, 1024), (37, 41), (300, 128)])
def test_fbp_segments_hold_every_bin(n, px, rows, seg):
    """The staged bins of a block of 64 columns, from the lowest corner's bin to
    the highest one's right neighbour (float32, the kernel's operations)."""
    rng = np.random.default_rng(n)
    th = np.concatenate([np.linspace(0, 2 * np.pi, 181), rng.uniform(0, 2 * np.pi, 60)])
    C, S = np.cos(th).astype(f32)[:, None, None], np.sin(th).astype(f32)[:, None, None]
    tiles = [(x, y) for x in range((n + 63) // 64) for y in range((n + rows - 1) // rows)]
    for tx, ty in [tiles[0], tiles[-1]] + [tiles[i] for i in rng.integers(0, len(tiles), 12)]:
        X = np.minimum(tx * 64 + np.arange(64), n - 1).astype(f32) - f32(n * 0.5)
        Y = np.minimum(ty * rows + np.arange(rows), n - 1).astype(f32) - f32(n * 0.5)
        u = (((X[None, None, :] * C).astype(f32) - (Y[None, :, None] * S).astype(f32)).astype(f32) + f32(px * 0.5)).astype(f32)
        b = np.floor(u)
        lo = b[:, [0, 0, -1, -1], [0, -1, 0, -1]].min(1)
        hi = b[:, [0, 0, -1, -1], [0, -1, 0, -1]].max(1)
        assert (b >= lo[:, None, None]).all() and (b <= hi[:, None, None]).all()
        assert (hi - lo + 2).max() <= seg
