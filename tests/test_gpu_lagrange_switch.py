"""VLP4D_LAG_FUSED is read when a Lagrange context is created: changed between
creation and a step, in either direction, it leaves the context's passes as
they are (the density partials are sized for them), and the steps still match
the oracle.

The grids have several vx runs per vy in the fused pass, so that its density
partials are more planes than the separate kernels'.  Three steps differ from
the oracle by some tens of roundings: 1e-12, the solver's bar.
"""
import math

import pytest

from conftest import relmax, sld_box

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [(16, 12, 40, 10), (64, 33, 24, 11), (129, 65, 12, 10)])
@pytest.mark.parametrize("at_creation,at_step", [("0", None), ("0", "1"), (None, "0")])
def test_switch_is_fixed_at_creation(vlp, orc, monkeypatch, n, at_creation, at_step):
    def switch(v):
        if v is None:
            monkeypatch.delenv("VLP4D_LAG_FUSED", raising=False)
        else:
            monkeypatch.setenv("VLP4D_LAG_FUSED", v)

    args = sld_box(n, vmax=6.0, dt=0.11, nbiter=3, idcase=10, lx=4 * math.pi)
    st = orc.LagState(orc.make_config(*args))
    st.step(3)
    switch(at_creation)
    with vlp.Vlp4d(vlp.VlpConfig.make(*args), scheme=vlp.SCHEME_LAGRANGE) as sim:
        switch(at_step)
        # before any step: a context that followed the switch would write past its buffer
        assert sim.kernel_variants() & 1 == (0 if at_creation == "0" else 1)
        sim.step(1)
        sim.step(2)
        assert relmax(sim.get_f(), st.f()) < 1e-12
        assert relmax(sim.buffer(vlp.BUF_EX), st.field(1)) < 1e-12
        assert relmax(sim.diags()["nrj"][1:], st.diags()["nrj"][1:]) < 1e-12
    st.close()
