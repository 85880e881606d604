"""The one-slice alignment adjoint at six and eight blocks a compute unit: sides
around the two lines of that choice (2049 and 2304 tiles of 16 x 16 pixels on 256
compute units).  A slice's sum does not depend on it, nor on how many slices are
staged together: equal to the same slice in a pair, bit for bit."""
import numpy as np
import pytest

from _util import dev, host, say

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx,ny", [(720, 720), (736, 729), (768, 768), (784, 760), (1024, 529)])
def test_one_slice_equals_a_pair(ctx, nx, ny):
    pa, px = 37, 500
    rng = np.random.default_rng(nx + ny)
    ctx.set_geometry(nx, px, pa, 1, ny=ny, angles_deg=(np.arange(pa) * (180.0 / pa) + 0.21).astype(np.float32))
    y = dev(rng.normal(0.0, 1.0, (2, pa, px)).astype(np.float32))
    shifts = dev(rng.normal(0.0, 2.0, pa).astype(np.float32))
    say("adjoint rounds", nx, ny)
    pair, one = dev(np.zeros((2, ny, nx))), dev(np.zeros((1, ny, nx)))
    ctx.align_adjoint(y, shifts, 0.4, pair)
    for z in range(2):
        ctx.align_adjoint(y[z:z + 1].contiguous(), shifts, 0.4, one)
        assert np.array_equal(host(one)[0], host(pair)[z]), z
