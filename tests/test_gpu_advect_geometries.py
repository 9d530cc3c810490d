"""The 4-D advection over the geometries its dispatch distinguishes, against
the oracle.

The tolerance is that of the whole-step parity tests: a step sums 256 products
of weights (positive, sum 1) per cell and solves four lines, so two steps
differ from the oracle by some hundred roundings of the result's magnitude,
1e-14; 1e-12 is asserted, as elsewhere.
"""
import math

import numpy as np
import pytest

from conftest import relmax, sld_box

pytestmark = pytest.mark.gpu


def _run(vlp, orc, n, steps=2, vmax=6.0, alpha=0.4, precision=64):
    """Steps of a strongly perturbed f (both signs of Ex and Ey everywhere)
    from the library and the oracle."""
    lx = 4 * math.pi
    dt = 0.5 * (lx / max(n[0], n[1])) / vmax
    args = sld_box(n, vmax=vmax, dt=dt, nbiter=steps, idcase=10, lx=lx)
    cfg = vlp.VlpConfig.make(*args)
    x = np.arange(n[0]) * cfg.dx[0]
    y = np.arange(n[1]) * cfg.dx[1]
    vx = cfg.minPhy[2] + np.arange(n[2]) * cfg.dx[2]
    vy = cfg.minPhy[3] + np.arange(n[3]) * cfg.dx[3]
    sp = 1 + alpha * np.cos(0.5 * x + 0.3)[None, :] + alpha * np.sin(0.5 * y + 0.2)[:, None]
    f0 = (np.exp(-0.5 * (vx[None, :] ** 2 + vy[:, None] ** 2)) / (2 * math.pi))[:, :, None, None] * sp[None, None]
    st = orc.State(orc.make_config(*args))
    st.set_f(f0)
    st.step(steps)
    ref, nrj = st.f_interior(), st.diags()["nrj"][1:]
    st.close()
    with vlp.Vlp4d(cfg, precision=precision) as sim:
        sim.set_f(f0)
        sim.step(steps)
        return relmax(sim.get_f(), ref), relmax(sim.diags()["nrj"][1:], nrj)


# A vy = 0 slab (even Nvy), whose feet have both y offsets and which two
# workgroups share: one and two vx tiles per wave, 8 tiles (XCD order), the
# smallest grid; odd Nvy has no such slab.
@pytest.mark.parametrize("n", [(16, 10, 10, 10), (16, 16, 16, 16), (32, 21, 16, 12), (64, 13, 12, 14), (32, 12, 14, 11)])
def test_slab_of_both_y_offsets(vlp, orc, n):
    ef, en = _run(vlp, orc, n)
    assert ef < 1e-12 and en < 1e-12


# Velocity displacements dt E / dv on both sides of one cell: below it a foot
# is streamed (with the clamp at the first velocity plane), beyond it the foot
# takes the direct gather (with the clamp at both ends).
@pytest.mark.parametrize("n,vmax", [((16, 10, 64, 64), 3.0), ((16, 16, 48, 20), 4.0), ((32, 12, 16, 90), 3.0)])
def test_velocity_displacement_beyond_a_cell(vlp, orc, n, vmax):
    ef, en = _run(vlp, orc, n, vmax=vmax)
    assert ef < 1e-12 and en < 1e-12


# Grids whose rows, tiles and planes do not divide evenly: rows of 4 k + 1, 2,
# 3 values (so that a plane's rows start 1 to 3 floats past a 16-byte
# boundary), a last vx tile reaching past Nvx, a last wave with few lanes,
# the longest rows.  In float a coefficient is stored to 2^-24 relative and is
# up to sqrt(3)^4 = 9 times f, so two steps differ by about 2 * 9 * 6e-8, and
# float interpolation adds some 10 roundings per step: 4e-6 is asserted.
RAGGED = [(61, 13, 11, 12), (17, 12, 13, 10), (90, 11, 21, 10), (51, 12, 19, 13), (251, 10, 11, 10), (10, 77, 10, 15)]


@pytest.mark.parametrize("n", RAGGED)
@pytest.mark.parametrize("precision,tol", [(64, 1e-12), (32, 4e-6), (33, 4e-6)])
def test_ragged_grids(vlp, orc, n, precision, tol):
    ef, en = _run(vlp, orc, n, precision=precision)
    assert ef < tol and en < tol


# Few workgroups: y goes in segments of one cell more than a quarter of the
# extent down to four cells, the last one shorter; many: one segment.
@pytest.mark.parametrize("n", [(16, 16, 10, 10), (16, 17, 10, 10), (16, 19, 12, 11), (10, 31, 10, 10), (32, 64, 10, 12),
                               (16, 13, 64, 66)])
def test_y_segments(vlp, orc, n):
    ef, en = _run(vlp, orc, n)
    assert ef < 1e-12 and en < 1e-12
