"""Reading CXY through vlp_get_buffer: the planes, stored with padding, come
back without it, in one piece (double, few floats) and in two (many floats),
and the call takes no host memory of the buffer's size beside the caller's.
"""
import math
import threading

import numpy as np
import psutil
import pytest

from conftest import relmax, sld_box

pytestmark = pytest.mark.gpu


# planes of (N0 + 4)(N1 + 4) values with every kind of padding to 16, none
# among them; sizes below and above the one from which floats are converted on
# the device
@pytest.mark.parametrize("n", [(12, 12, 10, 11), (13, 11, 12, 10), (28, 28, 14, 15), (45, 43, 37, 41), (44, 44, 40, 42)])
def test_cxy_is_the_same_in_every_precision(vlp, n):
    """Float storage rounds the two passes' coefficients (up to sqrt(3)^2 = 3
    times f) to 2^-24 each; a misplaced value would differ by its own size."""
    cfg = vlp.VlpConfig.make(*sld_box(n))
    rng = np.random.default_rng(sum(n))
    got = {}
    for precision in (64, 32):
        with vlp.Vlp4d(cfg, precision=precision) as sim:
            f = sim.get_f() if not got else start
            if not got:
                start = (f * (1 + 0.3 * rng.standard_normal(f.shape))).astype(np.float32).astype(np.float64)
            sim.set_f(start)
            sim.spline_xy()
            got[precision] = sim.buffer(vlp.BUF_CXY)
    assert got[64].shape == got[32].shape
    assert relmax(got[32], got[64]) < 2 * 3 * 2.0 ** -24
    assert np.array_equal(got[32], got[32].astype(np.float32))


@pytest.mark.parametrize("precision", [64, 32])
def test_cxy_takes_no_second_copy(vlp, precision):
    """A 64^4 CXY is 151 MB of doubles: the process may grow by those (the
    caller's array, touched by the copy) and some staging, not by twice them."""
    size = 68 * 68 * 64 * 64 * 8
    with vlp.Vlp4d(vlp.VlpConfig.make(*sld_box(64)), precision=precision) as sim:
        sim.spline_xy()
        host = np.empty(size // 8)
        proc = psutil.Process()
        base, peak, stop = proc.memory_info().rss, [0], threading.Event()

        def watch():
            while not stop.wait(0.0005):
                peak[0] = max(peak[0], proc.memory_info().rss)

        t = threading.Thread(target=watch)
        t.start()
        try:
            sim._check(sim.lib.vlp_get_buffer(sim.h, vlp.BUF_CXY, vlp._dptr(host), host.size))
        finally:
            stop.set()
            t.join()
    assert math.isfinite(host.sum())
    assert 0 < peak[0] - base < 1.5 * size
