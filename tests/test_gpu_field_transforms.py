"""The field solve's transforms over the factorisations of the extents (powers
of two, squares, two factors, primes and twice a prime, the smallest and the
longest), against numpy's FFT.

Each output is a sum of at most N + M products of a density of size 1 with
unit factors, N, M < 256, divided by k^2 >= 1/4: rounding of a few hundred
times 1e-16 of the field's maximum at worst, 1e-13; 1e-12 is asserted.
"""
import math

import numpy as np
import pytest

from conftest import relmax, sld_box

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx,ny", [(10, 11), (16, 25), (17, 10), (64, 121), (97, 22), (128, 127), (127, 128), (122, 94),
                                   (250, 251), (251, 15)])
def test_field_matches_fft(vlp, nx, ny):
    n, lx = (nx, ny, 10, 10), 4 * math.pi
    rng = np.random.default_rng(nx * 1000 + ny)
    with vlp.Vlp4d(vlp.VlpConfig.make(*sld_box(n, lx=lx))) as sim:
        f = rng.uniform(0.5, 1.5, n[::-1])
        sim.set_f(f)
        phi, ex, ey = (sim.buffer(b) for b in (vlp.BUF_RHO, vlp.BUF_EX, vlp.BUF_EY))
        dv = sim.cfg.dx[2] * sim.cfg.dx[3]
        d = sim.diags()
        da = sim.cfg.dx[0] * sim.cfg.dx[1]
    h = np.fft.rfft2(f.sum(axis=(0, 1)) * dv - 1)
    kx = np.arange(nx // 2 + 1)[None, :] * (2 * math.pi / lx)
    i = np.arange(ny)
    ky = np.where(i < ny // 2 + 1, i, i - ny)[:, None] * (2 * math.pi / lx)
    k2 = kx ** 2 + ky ** 2
    k2[0, 0] = 1
    h /= k2
    h[0, 0] = 0
    for got, spec in ((phi, h), (ex, -1j * kx * h), (ey, -1j * ky * h)):
        assert relmax(got, np.fft.irfft2(spec, s=(ny, nx))) < 1e-12
    assert abs(d["nrj"][0] - math.log(math.sqrt((ex ** 2 + ey ** 2).sum() * da))) < 1e-12
