"""Who decides how a side's slices run.  A schedule that the caller sets, and rows
asked for as set, hold for every slice of the side; the tuner's pick among
single-slice schedules does not take a stack off the interleaved kernels.  The
launches counted by the kernel timing tell the routes apart: a part that runs
interleaved and a part that runs singly are one projection each per subset, and
the images are those of the default route bit for bit."""
import numpy as np
import pytest
from ctrecon import Context

from _util import dev, host, say

pytestmark = pytest.mark.gpu


@pytest.fixture()
def own():
    c = Context(0)
    yield c
    c.close()


def _timed(c, call):
    c.set_kernel_timing(True)
    try:
        call()
        c.synchronize()
        return c.kernel_timing()[2]
    finally:
        c.set_kernel_timing(False)


def _angles(pa):
    return (np.arange(pa) * (180.0 / pa)).astype(np.float32)


def _stack(c, n, pa, dn):
    """(projection launches, images) of one iteration of one subset."""
    rng = np.random.default_rng(n + dn)
    x = dev(rng.uniform(0.2, 1.5, (dn, n, n)))
    y = dev(rng.uniform(0.0, 60.0, (dn, pa, n)))
    return _timed(c, lambda: c.osem_execution(x, y, 1)), host(x)


def test_a_schedule_that_is_set_runs(own):
    n, pa, dn = 520, 160, 5                      # four slices interleaved, one left over
    own.set_geometry(n, n, pa, 1, angles_deg=_angles(pa))
    say("set schedule", n, dn)
    launches, want = _stack(own, n, pa, dn)
    assert launches == 2
    own.set_schedule(n, 0, 4, 4, fp_tile=44)
    launches, got = _stack(own, n, pa, dn)
    assert launches == 1 and np.array_equal(got, want)
    own.set_schedule(n, 0, 4, 8)                 # the defaults: as at first
    assert _stack(own, n, pa, dn)[0] == 2
    own.set_adaptive_rows(False)
    launches, got = _stack(own, n, pa, dn)
    assert launches == 1 and np.array_equal(got, want)
    own.set_adaptive_rows(True)
    assert _stack(own, n, pa, dn)[0] == 2


def test_a_schedule_that_is_set_runs_in_a_batch(own):
    pa, sides = 240, [256] * 16 + [200] * 4
    own.set_geometry(256, 256, pa, 1, angles_deg=_angles(pa))
    rng = np.random.default_rng(3)
    x0 = [rng.uniform(0.2, 1.5, (n, n)) for n in sides]
    prjs = [dev(rng.uniform(0.0, 60.0, (pa, n))) for n in sides]
    say("set schedule in a batch")

    def run():
        imgs = [dev(v) for v in x0]
        return _timed(own, lambda: own.osem_batched(imgs, prjs, 1)), [host(v) for v in imgs]

    launches, want = run()
    assert launches == 1                         # all interleaved
    own.set_schedule(200, 0, 4, 4, fp_tile=32)
    launches, got = run()
    assert launches == 2 and all(np.array_equal(a, b) for a, b in zip(got, want))
    own.set_adaptive_rows(False)
    launches, got = run()
    assert launches == 2 and all(np.array_equal(a, b) for a, b in zip(got, want))    # two schedules, both single


def test_the_tuners_pick_keeps_stacks_interleaved(own):
    """A direct gather sums a ray in another order: a stack that went over to it would
    have other images.  On the smallest sides it is the tuner's usual pick."""
    picks = {}
    for n in (8, 16, 32):
        pa, dn = 120 if n < 32 else 60, 704 if n < 32 else 1200
        own.set_geometry(n, n, pa, 1, angles_deg=_angles(pa))
        say("tuned", n, dn)
        want = _stack(own, n, pa, dn)[1]
        picks[n] = own.autotune(n)["fp_rays"]
        launches, got = _stack(own, n, pa, dn)
        assert launches == 1 and np.array_equal(got, want), picks
    print(f"[autotune] rays per wave by side (0: LDS tiles): {picks}", flush=True)
