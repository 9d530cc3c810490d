"""vlp_field_solve of a float f that is aligned to its elements only: the
density pass takes four, two or one points per thread by the plane's size
alone, and its loads are those of the same f at an aligned address.  Same
values in the same order: the results are equal bit for bit.
"""
import numpy as np
import pytest

from conftest import sld_box

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [(10, 10, 12, 11), (12, 11, 13, 10), (11, 10, 15, 13), (11, 13, 10, 12)])
@pytest.mark.parametrize("entry", ["field_solve", "field_solve_noalloc"])
def test_float_f_at_any_element(vlp, n, entry):
    from hip_buffers import DeviceArray
    vlp.load()
    gc = vlp.VlpConfig.make(*sld_box(n))
    rng = np.random.default_rng(sum(n))
    f = rng.uniform(0.5, 1.5, n[::-1]).astype(np.float32).ravel()
    n2 = n[0] * n[1]
    out = []
    for shift in range(4):
        fd = DeviceArray.of(np.concatenate([np.full(shift, np.nan, np.float32), f, np.full(4, np.nan, np.float32)]))
        phi, ex, ey, diag = DeviceArray(8 * n2), DeviceArray(8 * n2), DeviceArray(8 * n2), DeviceArray(8 * 5)
        getattr(vlp, entry)(gc, fd.addr + 4 * shift, 32, phi.addr, ex.addr, ey.addr, diag.addr)
        out.append(np.concatenate([phi.get(np.float64, n2), ex.get(np.float64, n2), ey.get(np.float64, n2),
                                   diag.get(np.float64, 5)]))
        for d in (fd, phi, ex, ey, diag):
            d.free()
    assert np.all(np.isfinite(out[0])) and np.abs(out[0][:n2]).max() > 0
    for o in out[1:]:
        assert np.array_equal(o, out[0])
