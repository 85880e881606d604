"""The rotation-centre shift of one, two and three candidates in a context that has
held no more before (the device table of shifts is then as small as the upload)."""
import numpy as np
import pytest
from ctrecon import Context

import oracle as O
from _util import dev, host, say

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("cnt", [1, 2, 3])
def test_few_candidates_in_a_fresh_context(cnt):
    pa, px = 5, 40
    ctx = Context(0)
    try:
        ctx.set_geometry(px, px, pa, 1, angles_deg=np.arange(pa, dtype=np.float32) * 36.0)
        prj = np.random.default_rng(cnt).uniform(-1.0, 2.0, (pa, px)).astype(np.float32)
        say("few candidates", cnt)
        for _ in range(2):
            out = dev(np.zeros((cnt, pa, px)))
            ctx.op("rot_center_shift", dev(prj), out, cnt, -2.35, 1.7)
            assert np.array_equal(host(out), O.rot_center_shift(O.geom(px, px, pa, ss=1), prj, cnt, -2.35, 1.7))
    finally:
        ctx.close()
