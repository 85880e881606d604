"""The choice between quads and single slices, from the library's own functions on the
host: stacks that the GPU tests mean to run as quads do so, and batches of several
sides stay single where quads would lose."""
import numpy as np

import _quads
import test_gpu_coupled_stacks
import test_gpu_quads
from test_gpu_quads import _angles


def _rows(test, names):
    for mark in test.pytestmark:
        if mark.name == "parametrize" and mark.args[0] == names:
            return mark.args[1]
    raise KeyError(names)


def test_stacks_meant_as_quads():
    for nx, ny, px, pa, ss, dn, kind in _rows(test_gpu_quads.test_quads_equal_single_slices, "nx,ny,px,pa,ss,dn,kind"):
        if (nx, kind) == (512, "wide"):
            continue                             # angles too far apart to share windows: single slices
        ang = _angles(kind, pa, np.random.default_rng(nx + 3 * ny + px))
        assert _quads.stack_quads(nx, ny, px, pa, ss, dn, ang.astype(np.float32)) >= dn - 1, (nx, kind)
    for nx, ny, px, pa, ss, dn in test_gpu_coupled_stacks.CASES[:3]:
        assert _quads.stack_quads(nx, ny, px, pa, ss, dn, np.arange(pa) * (180.0 / pa)) >= dn - 1, nx


def test_batches():
    assert _quads.batch_quads([64] * 8 + [200] * 13 + [129] * 14 + [257] * 7 + [90] * 2 + [301], 120) == 41
    assert _quads.batch_quads([135] * 6 + [137] * 4 + [1003] * 3, 62) == 0        # 604 blocks
    assert _quads.batch_quads([445] * 8 + [524] * 12 + [713] * 4, 30) == 24       # 795
    assert _quads.batch_quads([1024] * 17, 45) == 16
    assert _quads.batch_quads([512] * 8, 80) == 8


def test_angles_far_apart():
    def turn(pa):
        return np.arange(pa) * (180.0 / pa)
    assert _quads.stack_quads(2048, 2048, 2048, 50, 1, 4, turn(50)) == 4        # rims 64 texels apart
    assert _quads.stack_quads(1024, 1024, 1024, 20, 1, 24, turn(20)) == 0       # 80
    assert _quads.align_quads(2048, 2048, 2048, 80, 4, turn(80)) == 4           # 40
    assert _quads.align_quads(2048, 2048, 2048, 60, 4, turn(60)) == 0           # 54
