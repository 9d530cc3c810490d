"""The adjoint step's kernels over the grids their launches distinguish, against
the per-cell form (VLP4D_ADJ_BLOCK=0): blocks of 2^3 and of 4^3 cells in
(y, vx, vy) with remainders of each, x in one and several extents, planes and
lines that are no multiple of a wave, columns that leave a wave part idle, long
lines.

Both forms sum the same terms in different orders, and the blocked one rounds
each to 2^-50 of the largest cotangent: 1e-12 of the gradient's largest entry.
"""
import numpy as np
import pytest

from conftest import sld_box

pytestmark = pytest.mark.gpu

GRIDS = [(10, 10, 10, 10), (33, 11, 13, 10), (17, 12, 41, 15), (32, 30, 22, 21), (65, 14, 17, 18), (13, 67, 10, 33),
         (70, 21, 24, 23), (129, 10, 11, 10), (10, 251, 10, 10), (10, 10, 130, 12)]


@pytest.mark.parametrize("n", GRIDS)
def test_blocked_adjoint_matches_per_cell_form(vlp, monkeypatch, n):
    vmax, lx = 6.0, 12.0
    cfg = vlp.VlpConfig.make(*sld_box(n, vmax=vmax, dt=0.5 * (lx / max(n[0], n[1])) / vmax, nbiter=10, idcase=10,
                                      lx=lx))
    rng = np.random.default_rng(sum(n))
    out = []
    for blk in ("1", "0"):
        monkeypatch.setenv("VLP4D_ADJ_BLOCK", blk)
        with vlp.Vlp4d(cfg) as sim:
            f0 = sim.get_f()
            if not out:
                f0 = f0 * (1 + 0.1 * rng.standard_normal(f0.shape))
                g = rng.standard_normal(f0.shape)
                start = f0
            sim.set_f(start)
            out.append(sim.adjoint_step(g))
    a, b = out
    assert np.abs(b).max() > 0.1
    np.testing.assert_allclose(a, b, rtol=0, atol=1e-12 * np.abs(b).max())
