"""The Lagrange solver's fused x/2, y/2 pass over the planes its dispatch
distinguishes, against the oracle: 16 and 32 points per lane, one and several
64-line groups, remainders of both, odd rows, planes of up to 16 waves, planes
that do not fit (separate kernels); runs of several steps in one call, whose
neighbouring pairs are one pass, against the same steps one call each.

Six-point stencils have weights of absolute sum below 1.7; a step is six of
them per cell, so three steps differ by some tens of roundings from the
oracle's: 1e-12 is the solver's bar, 1e-13 asserted between the two call
patterns.
"""
import math

import numpy as np
import pytest

from conftest import relmax, sld_box

pytestmark = pytest.mark.gpu

PLANES = [(10, 10, 10, 11), (16, 16, 12, 10), (17, 33, 10, 13), (64, 64, 10, 12), (65, 63, 11, 10), (61, 130, 10, 10),
          (97, 66, 13, 10), (127, 128, 10, 10), (100, 160, 10, 10), (66, 245, 10, 10), (251, 20, 10, 10),
          (140, 150, 10, 10)]


@pytest.mark.parametrize("n", PLANES)
def test_planes_match_oracle(vlp, orc, n):
    steps, vmax, lx = 3, 6.0, 4 * math.pi
    args = sld_box(n, vmax=vmax, dt=0.11, nbiter=steps, idcase=10, lx=lx)
    rng = np.random.default_rng(n[0] + n[1])
    st = orc.LagState(orc.make_config(*args))
    f0 = st.f() * (1 + 0.1 * rng.standard_normal(st.f().shape))
    st.set_f(f0)
    st.step(steps)
    got = {}
    for calls in ((steps,), (1,) * steps):
        with vlp.Vlp4d(vlp.VlpConfig.make(*args), scheme=vlp.SCHEME_LAGRANGE) as sim:
            sim.set_f(f0)
            for k in calls:
                sim.step(k)
            assert sim.iter == steps
            got[len(calls)] = sim.get_f(), sim.diags()["nrj"], sim.buffer(vlp.BUF_EX)
    f, nrj, ex = got[1]
    assert relmax(f, st.f()) < 1e-12
    assert relmax(nrj[1:], st.diags()["nrj"][1:]) < 1e-12
    assert relmax(ex, st.field(1)) < 1e-12
    for a, b in zip(got[1], got[steps]):
        assert relmax(a, b) < 1e-13
    st.close()
