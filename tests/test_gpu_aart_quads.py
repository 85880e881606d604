"""AART of stacks that run as quads: enough subsets in all, or enough backprojection
blocks, for the backprojection of the sinograms that it begins with.  Equal to one
slice at a time bit for bit, at the sizes of the coupled stacks' edges."""
import numpy as np
import pytest

import _quads
from _util import dev, host, say
from test_gpu_coupled_stacks import CASES, _inputs


def _angles(pa):
    return (np.arange(pa) * (180.0 / pa)).astype(np.float32)


QUADS = [c + (4,) for c in CASES[:3]] + [(193, 130, 180, 108, 3, 46, 1)]       # the last by its blocks


def test_they_run_as_quads():
    for nx, ny, px, pa, ss, dn, it in QUADS:
        assert _quads.stack_quads(nx, ny, px, pa, ss, dn, _angles(pa), passes=ss * it) >= dn - 1
        assert ss * it >= 8 or (nx, ny) == (193, 130)
    nx, ny, px, pa, ss, dn = CASES[0]
    assert _quads.stack_quads(nx, ny, px, pa, ss, dn, _angles(pa), passes=ss * 2) == 0


@pytest.mark.gpu
@pytest.mark.parametrize("nx,ny,px,pa,ss,dn,it", QUADS)
def test_aart_quads_equal_single_slices(ctx, nx, ny, px, pa, ss, dn, it):
    x0, y = _inputs(ctx, nx, ny, px, pa, ss, dn, mode=2)
    say("aart quads", nx, ny, px, pa, ss, dn, it)
    got = dev(x0)
    ctx.aart_execution(got, dev(y), it)
    for z in sorted({0, 1, dn // 2, dn - 3, dn - 2, dn - 1}):
        one = dev(x0[z:z + 1])
        ctx.aart_execution(one, dev(y[z:z + 1]), it)
        assert np.array_equal(host(one)[0], host(got)[z]), z
