"""Quads whose blocks walk their two angles one after the other, over many chunks and
bands of large images: angle tables that lie close on average, as the rule asks, but
whose neighbours now and then differ by tens of degrees, by a half turn (the other
direction) or by a quarter turn (the other image copy).  The first test holds the
tables to that with the bounds' own restatement; images and rows equal those of
single slices bit for bit."""
import numpy as np
import pytest

import _quads
import test_quad_bounds as tb
from _util import dev, host, say


def _angles(kind, pa):
    a = np.arange(pa) * (180.0 / pa)
    k = np.arange(pa)
    if kind == "jumps":
        a += 25.0 * (k % 5 == 2)
    elif kind == "half turns":
        a += 180.0 * (k % 3 == 0)
    else:
        a += 90.0 * (k % (20 if pa < 200 else 60) == 7)
    return a.astype(np.float32)


CASES = [
    # nx, ny, px, pa, dn, kind
    (512, 512, 512, 90, 12, "jumps"), (512, 512, 512, 90, 11, "half turns"), (512, 512, 530, 91, 12, "quarter turns"),
    (700, 333, 650, 120, 8, "half turns"), (1100, 1100, 1100, 240, 4, "quarter turns"),
]


def test_tables_stay_quads_and_refuse_to_share():
    for nx, ny, px, pa, dn, kind in CASES:
        ang = _angles(kind, pa)
        assert _quads.stack_quads(nx, ny, px, pa, 1, dn, ang) == dn, (nx, kind)
        rad = ang.astype(np.float64) * np.pi / 180.0
        c, s = np.cos(rad).astype(np.float32), np.sin(rad).astype(np.float32)
        ch = (px // tb.LT) // 2
        share = [tb._share([tb._Ray(nx, ny, px, c[j + a], s[j + a], ch, False) for a in range(2)])
                 for j in range(0, min(pa - 1, 60), 2)]
        assert 0 < sum(not v for v in share) < 0.9 * len(share), (nx, kind, share)


@pytest.mark.gpu
@pytest.mark.parametrize("nx,ny,px,pa,dn,kind", CASES)
def test_images_equal_single_slices(ctx, nx, ny, px, pa, dn, kind):
    rng = np.random.default_rng(nx + 3 * ny + px)
    ctx.set_geometry(nx, px, pa, 1, ny=ny, angles_deg=_angles(kind, pa))
    x0 = rng.uniform(0.2, 1.5, (dn, ny, nx)).astype(np.float32)
    y = rng.uniform(0.0, 60.0, (dn, pa, px)).astype(np.float32)
    say("quad walks", nx, ny, px, pa, dn, kind)
    a = dev(x0)
    ctx.osem_execution(a, dev(y), 2)
    got = host(a)
    for z in (0, 1, dn - 2, dn - 1):
        b = dev(x0[z:z + 1])
        ctx.osem_execution(b, dev(y[z:z + 1]), 2)
        assert np.array_equal(got[z], host(b)[0]), z


@pytest.mark.gpu
@pytest.mark.parametrize("kind", ["jumps", "half turns", "quarter turns"])
def test_alignment_rows_equal_single_layers(ctx, kind):
    n, px, pa, dn = 400, 333, 361, 8
    ang = _angles(kind, pa)
    assert _quads.align_quads(n, n, px, pa, dn, ang) == dn
    rng = np.random.default_rng(len(kind))
    ctx.set_geometry(n, px, pa, 1, angles_deg=ang)
    x = dev(rng.uniform(-0.5, 1.0, (dn, n, n)).astype(np.float32))
    sh = rng.normal(0.0, 4.0, pa).astype(np.float32)
    sh[::9] *= 30.0
    shifts = dev(sh)
    say("quad walks, alignment", kind)

    def forward(img):
        p, d = (dev(np.full((img.shape[0], pa, px), 7.0, np.float32)) for _ in range(2))
        ctx.align_forward_deriv(img, shifts, 0.7, p, d)
        ctx.synchronize()
        return host(p), host(d)

    got = forward(x)
    for z in (0, 3, dn - 1):
        one = forward(x[z:z + 1].contiguous())
        assert np.array_equal(got[0][z], one[0][0]) and np.array_equal(got[1][z], one[1][0]), z
