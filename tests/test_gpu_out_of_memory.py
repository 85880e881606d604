"""Calls whose workspace does not fit the device: they report out of memory, again
when called again, leave the caller's buffers as they were, and the next call that
fits runs.  The stacks are nominally large (sides of 16384, a detector of a few bins)
so that the first allocation that fails is far beyond any device's memory; nothing
runs on the images, which are small buffers here."""
import ctypes as C

import numpy as np
import pytest
from ctrecon import Context
from ctrecon._lib import Slice

from _util import dev, host, say

pytestmark = pytest.mark.gpu
CTR_OUT_OF_MEMORY = 4
SIDE, COUNT = 16384, 400                     # 400 padded images of 1.1 GB


@pytest.fixture()
def own():
    c = Context(0)
    yield c
    c.close()


def _small_run(c):
    n, pa, ss = 64, 24, 4
    ang = (np.arange(pa) * (180.0 / pa)).astype(np.float32)
    c.set_geometry(n, n, pa, ss, angles_deg=ang)
    x = dev(np.ones((1, n, n)))
    c.osem_execution(x, dev(np.random.default_rng(1).uniform(0.0, 9.0, (1, pa, n))), 1)
    c.synchronize()
    assert np.isfinite(host(x)).all() and not (host(x) == 1.0).all()


def test_batched_list_too_large(own):
    pa, ss = 4, 2
    own.set_geometry(64, 64, pa, ss, angles_deg=np.arange(pa, dtype=np.float32) * 45.0)
    x, y = dev(np.ones((64, 64))), dev(np.ones((pa, 64)))
    slices = (Slice * COUNT)(*[Slice(SIDE, x.data_ptr(), y.data_ptr()) for _ in range(COUNT)])
    say("batched list too large")
    for _ in range(2):
        st = own.lib.ctr_osem_batched(own.h, slices, COUNT, 1, 0)
        assert st == CTR_OUT_OF_MEMORY, own.lib.ctr_last_error(own.h)
    assert (host(x) == 1.0).all()
    # a list that fits runs after it
    imgs, prjs = [dev(np.ones((64, 64)))], [dev(np.full((pa, 64), 7.0))]
    own.osem_batched(imgs, prjs, 1, use_graph=True)
    own.synchronize()
    assert not (host(imgs[0]) == 1.0).all()
    _small_run(own)


@pytest.mark.parametrize("driver", ["ctr_osem_execution", "ctr_fista_osem_execution", "ctr_aart_execution"])
def test_stack_too_large_keeps_its_sinograms(own, driver):
    pa, ss, px = 4, 2, 8
    own.set_geometry(SIDE, px, pa, ss, mode=2, correction_mode=1, angles_deg=np.arange(pa, dtype=np.float32) * 45.0)
    x, y0 = dev(np.ones((64, 64))), np.random.default_rng(2).uniform(1.0, 9.0, (COUNT, pa, px)).astype(np.float32)
    y = dev(y0)
    say("stack too large", driver)
    args = [own.h, C.c_void_p(x.data_ptr()), C.c_void_p(y.data_ptr()), COUNT, 1] + ([1] if driver != "ctr_aart_execution" else [])
    for _ in range(2):
        st = getattr(own.lib, driver)(*args)
        assert st == CTR_OUT_OF_MEMORY, own.lib.ctr_last_error(own.h)
        own.synchronize()
        assert np.array_equal(host(y), y0)
    _small_run(own)
