"""The fused x/y spline and half-step kernel over the workgroup sizes and plane
groups its dispatch distinguishes, against the oracle: 128, 256 and 512 lanes,
lines that fill them and that leave some idle, one plane per group and several,
a shorter last group, more workgroups than the chip holds at once.

The tolerance is that of the whole-step parity tests: two steps differ from the
oracle by some hundred roundings of the result's magnitude, 1e-14; 1e-12 is
asserted, as elsewhere.  In float a coefficient is stored to 2^-24 relative and
is up to sqrt(3)^4 = 9 times f, so two steps differ by about 2 * 9 * 6e-8, and
float interpolation adds some 10 roundings per step: 4e-6.
"""
import math

import numpy as np
import pytest

from conftest import relmax, sld_box

pytestmark = pytest.mark.gpu

GRIDS = [(10, 10, 12, 11), (13, 14, 21, 10), (25, 23, 33, 12), (28, 31, 13, 10),  # 128 lanes
         (31, 33, 11, 10), (36, 36, 10, 14), (20, 60, 15, 10), (45, 37, 17, 11), (61, 28, 10, 10),  # 256
         (11, 100, 10, 10), (120, 10, 11, 10), (61, 50, 10, 12), (65, 45, 11, 10),  # 256, 512
         (10, 11, 61, 90), (24, 25, 64, 67)]  # groups of several planes


@pytest.mark.parametrize("n", GRIDS)
@pytest.mark.parametrize("precision,tol", [(64, 1e-12), (32, 4e-6), (33, 4e-6)])
def test_steps_match_oracle(vlp, orc, n, precision, tol):
    steps, vmax, lx = 2, 6.0, 4 * math.pi
    args = sld_box(n, vmax=vmax, dt=0.5 * (lx / max(n[0], n[1])) / vmax, nbiter=steps, idcase=10, lx=lx)
    rng = np.random.default_rng(sum(n))
    st = orc.State(orc.make_config(*args))
    f0 = st.f_interior() * (1 + 0.1 * rng.standard_normal(n[::-1]))
    st.set_f(f0)
    st.step(steps)
    with vlp.Vlp4d(vlp.VlpConfig.make(*args), precision=precision) as sim:
        assert sim.kernel_variants() & 4096
        sim.set_f(f0)
        sim.step(steps)
        assert relmax(sim.get_f(), st.f_interior()) < tol
        assert relmax(sim.diags()["nrj"][1:], st.diags()["nrj"][1:]) < tol
    st.close()
