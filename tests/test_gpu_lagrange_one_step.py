"""Lagrange steps one call each and several per call over the planes that the
x/2, y/2 pass's forms distinguish beyond those of whole 64-line groups: lanes
along the segments of few lines (one and several segments per wave, remainders
of both axes, no lane idle), single pairs with 16 points and no density sums,
the sizes on either side of each; runs of one plane and of several.

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

# flat lanes: thin planes, squares between the grouped form's sizes, 8 full waves
FLAT = [(10, 251, 10, 13), (251, 10, 11, 10), (16, 160, 12, 10), (160, 16, 10, 11), (200, 21, 10, 10),
        (68, 68, 10, 12), (67, 75, 11, 10), (64, 128, 12, 10), (128, 64, 10, 10), (100, 10, 10, 12), (11, 128, 12, 10),
        (31, 33, 10, 11)]
# 32 points per lane for the joined pairs, 16 for single ones
WIDE = [(90, 90, 10, 10), (100, 91, 13, 10), (129, 65, 10, 11), (65, 129, 10, 10), (128, 128, 10, 10), (89, 96, 12, 10)]
# the run lengths: one plane, a few, a shorter last run
RUNS = [(10, 10, 23, 11), (16, 16, 24, 60), (24, 17, 41, 76), (33, 20, 50, 90)]


@pytest.mark.parametrize("n", FLAT + WIDE + RUNS)
def test_one_step_calls_match_oracle(vlp, orc, n):
    steps, vmax, lx = 3, 6.0, 4 * math.pi
    args = sld_box(n, vmax=vmax, dt=0.11, nbiter=steps, idcase=10, lx=lx)
    rng = np.random.default_rng(n[0] + 3 * n[1])
    st = orc.LagState(orc.make_config(*args))
    f0 = st.f() * (1 + 0.1 * rng.standard_normal(st.f().shape))
    st.set_f(f0)
    st.step(steps)
    got = []
    for calls in ((1,) * steps, (steps,)):
        with vlp.Vlp4d(vlp.VlpConfig.make(*args), scheme=vlp.SCHEME_LAGRANGE) as sim:
            assert sim.kernel_variants() & 1
            sim.set_f(f0)
            for k in calls:
                sim.step(k)
            got.append((sim.get_f(), sim.diags()["nrj"], sim.buffer(vlp.BUF_EX)))
    f, nrj, ex = got[0]
    assert relmax(f, st.f()) < 1e-12
    assert relmax(nrj[1:], st.diags()["nrj"][1:]) < 1e-12
    assert relmax(ex, st.field(1)) < 1e-12
    for a, b in zip(*got):
        assert relmax(a, b) < 1e-13
    st.close()
