"""Float spline lines that four lanes of the line kernel divide evenly take it
or the tiles by the bytes a pass writes: C4 on either side of that size, by the
default choice and by the line kernel alone (VLP4D_SPLINE_TILE=0).

The two kernels sum in other orders; each of the two passes stores to 2^-24 of
coefficients up to sqrt(3)^4 = 9 times f: 2 * 9 * 2^-24 of the maximum.
"""
import numpy as np
import pytest

from conftest import relmax, sld_box

pytestmark = pytest.mark.gpu


# both passes below 100 MB (line kernel), above (tiles), and on either side;
# planes that are no whole 64-byte blocks
@pytest.mark.parametrize("n", [(52, 52, 72, 72), (72, 72, 72, 72), (64, 64, 68, 72), (31, 29, 108, 124), (41, 43, 108, 100)])
def test_four_lane_lengths(vlp, monkeypatch, n):
    cfg = vlp.VlpConfig.make(*sld_box(n))
    rng = np.random.default_rng(sum(n))
    out = []
    for tile in (None, "0"):
        if tile is not None:
            monkeypatch.setenv("VLP4D_SPLINE_TILE", tile)
        with vlp.Vlp4d(cfg, precision=32) as sim:
            if not out:
                f0 = sim.get_f() * (1 + 0.3 * rng.standard_normal(n[::-1]))
            sim.set_f(f0)
            sim.spline_xy()
            sim.spline_vxvy()
            out.append(sim.buffer(vlp.BUF_C4))
    assert np.abs(out[1]).max() > 0
    assert relmax(out[0], out[1]) < 2 * 9 * 2.0 ** -24
