"""The spline passes over line lengths of every kind -- whole chunks per lane,
a shorter last chunk (from one to all but one of its values repeated), one lane
per line, lanes without a chunk, lines and planes past the tiled kernels -- and
planes that do and do not fill whole 64-byte blocks: CXY and C4 against the
oracle.

The recursions damp by |alpha| = 0.27 per point, so a coefficient carries some
tens of roundings of at most sqrt(3)^4 = 9 times f: 1e-13 of the maximum, the
bar of the phase tests.  Float storage rounds each of four passes to 2^-24 of
coefficients up to that size.
"""
import numpy as np
import pytest

from conftest import relmax, sld_box

pytestmark = pytest.mark.gpu

LENGTHS = [(10, 11, 12, 13), (17, 33, 11, 23), (45, 50, 10, 10), (61, 77, 10, 10), (10, 10, 65, 75), (10, 11, 91, 101),
           (11, 13, 127, 128), (113, 90, 10, 10), (150, 130, 10, 10), (11, 10, 129, 160), (16, 20, 68, 72),
           (37, 97, 76, 21), (128, 31, 14, 49)]


@pytest.mark.parametrize("n", LENGTHS)
def test_line_lengths_match_oracle(vlp, orc, n):
    args = sld_box(n)
    oc = orc.make_config(*args)
    h = orc.init_case(oc)
    rng = np.random.default_rng(sum(n))
    orc.interior_of(h)[...] *= 1.0 + 0.3 * rng.standard_normal(orc.interior_shape(oc))
    f0 = np.ascontiguousarray(orc.interior_of(h))
    orc.exchange_halo(oc, h)
    orc.spline_xy(oc, h)
    cxy = h[3:-3, 3:-3, 1:-1, 1:-1].copy()  # positions -2..N+1 in x and y
    orc.spline_vxvy(oc, h)
    for precision, tol in ((64, 1e-13), (32, 4 * 9 * 2.0 ** -24)):
        with vlp.Vlp4d(vlp.VlpConfig.make(*args), precision=precision) as sim:
            sim.set_f(f0)
            sim.spline_xy()
            assert relmax(sim.buffer(vlp.BUF_CXY), cxy) < tol
            sim.spline_vxvy()
            assert relmax(sim.buffer(vlp.BUF_C4), orc.ext_view(h)) < tol
