"""The Lagrange solver's velocity passes against the oracle, over the grids the
dispatch of the fused pass distinguishes: planes that are no multiple of its
16 points, vx lengths with remainders of its 4 points per lane, up to
the 251 an axis may have, vy in one and many segments of 2 to 16 rows; fields
that shift lines by several cells, differently from point to point.

Two steps of a few tens of roundings, with shifts of up to some ten cells whose
rounding enters times the slope per cell of a 10 % noise: 1e-12.
"""
import math

import numpy as np
import pytest

from conftest import relmax, sld_box

pytestmark = pytest.mark.gpu

GRIDS = [(10, 10, 10, 10), (17, 11, 13, 35), (32, 32, 64, 33), (20, 13, 61, 40), (10, 12, 130, 49), (12, 11, 10, 129),
         (16, 10, 251, 18), (10, 10, 250, 10)]


@pytest.mark.parametrize("n", GRIDS)
def test_velocity_passes_match_oracle(vlp, orc, n):
    args = sld_box(n, vmax=6.0, dt=0.11, nbiter=4, idcase=10, lx=4 * math.pi)
    rng = np.random.default_rng(sum(n))
    st = orc.LagState(orc.make_config(*args))
    f0 = 30 * st.f() * (1 + 0.1 * rng.standard_normal(st.f().shape))
    st.set_f(f0)
    st.step(2)
    with vlp.Vlp4d(vlp.VlpConfig.make(*args), scheme=vlp.SCHEME_LAGRANGE) as sim:
        sim.set_f(f0)
        sim.step(2)
        assert relmax(sim.get_f(), st.f()) < 1e-12
        assert relmax(sim.buffer(vlp.BUF_EX), st.field(1)) < 1e-12
    st.close()
