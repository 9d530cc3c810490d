"""f, CXY and C4 between the host and float storage: set_f rounds each double
to the nearest float and get_f and get_buffer return the stored floats exactly,
for sizes with every remainder of the four values a lane converts, sizes that
go in one and in two pieces, and values at the ends of the float range."""
import numpy as np
import pytest

from conftest import relmax, sld_box

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [(10, 10, 10, 10), (11, 13, 11, 11), (11, 10, 11, 13), (11, 11, 13, 15), (64, 60, 50, 48)])
@pytest.mark.parametrize("precision", [32, 33])
def test_float_transfers_are_exact(vlp, n, precision):
    rng = np.random.default_rng(sum(n))
    f = rng.standard_normal(n[::-1]) * np.exp(rng.uniform(-20, 20, n[::-1]))
    f.ravel()[:5] = [0.0, -0.0, 3.0e38, 1.2e-38, 1.0 + 2.0 ** -24]
    f.ravel()[-1] = 1.0 + 3 * 2.0 ** -24
    with vlp.Vlp4d(vlp.VlpConfig.make(*sld_box(n)), precision=precision) as sim:
        sim.set_f(f)
        want = f.astype(np.float32).astype(np.float64)
        assert np.array_equal(sim.get_f(), want)
        assert np.array_equal(sim.buffer(vlp.BUF_F), want)


@pytest.mark.parametrize("n", [(16, 16, 12, 10), (13, 11, 12, 10)])
def test_float_coefficients_come_back_in_place(vlp, n):
    """CXY and C4 of float storage are those of double storage to the rounding
    of stored coefficients (four passes, each storing to 2^-24 of a value up to
    sqrt(3)^4 = 9 times f): a misplaced value would differ by its own size."""
    cfg = vlp.VlpConfig.make(*sld_box(n))
    got = {}
    for precision in (64, 32):
        with vlp.Vlp4d(cfg, precision=precision) as sim:
            sim.spline_xy()
            sim.spline_vxvy()
            got[precision] = sim.buffer(vlp.BUF_CXY), sim.buffer(vlp.BUF_C4)
    for a, b in zip(got[32], got[64]):
        assert a.shape == b.shape and relmax(a, b) < 4 * 9 * 2.0 ** -24
        assert np.array_equal(a, a.astype(np.float32))
