"""Single 2D steps with the energy curve (terms summed in the velocity launch) and
without it (a kernel of its own), in every tile height: the curve is summed by
tiles, so it agrees between them to rounding; nothing else depends on them.

Bars: fields and seismograms bit-exact with and without energy and between tile
heights; energy 1e-12 (double) / 1e-4 (float) rel-L2 between tile heights, and in 3D
between chunk depths.
"""
import numpy as np
import pytest

from gpu_runner import F2D, F3D, rel_l2
from seismic_cpml_amd import CpmlGpu
from seismic_cpml_amd import solver as S

pytestmark = pytest.mark.gpu

NSTEP = 10


def _run(n, order, prec, energy, tile, kchunk=0):
    ndim = len(n)
    nx, ny, nz = (*n, 1)[:3]
    dt = 0.4 * 10.0 / (4000.0 * 3 ** 0.5)
    rng = np.random.default_rng(sum(n))
    real = np.float32 if prec == 4 else np.float64
    shape = n[::-1]
    with CpmlGpu(ndim, order, prec, nx, ny, nz, 10.0, 10.0, 10.0, dt, 5, NSTEP) as s:
        rho = rng.uniform(2000, 2600, shape).astype(real)
        mu = (rho * 2000.0 ** 2).astype(real)
        s.set_medium((mu * 2).astype(real), mu, rho)
        s.set_pml(*(S.pml_profile(m, 10.0, dt, 5, 4000.0, 12.0, prec) for m in n))
        f = np.sin(np.arange(NSTEP)).astype(real)
        s.set_source(nx // 2, ny // 3, max(nz // 2, 1), f, -f)
        s.set_receivers(*[[1 + m // 3, m // 2] for m in n])
        for name in ("vx", "vy", "vz")[:ndim]:
            v = np.zeros(shape, real)
            v[(slice(2, -2),) * ndim] = rng.standard_normal([m - 4 for m in shape])
            s.set_field(name, v)
        if energy:
            s.set_energy(1)
        s.set_tile(tile)
        if kchunk:
            s.set_kchunk(kchunk)
        s.run()
        out = [s.field(k) for k in (F2D if ndim == 2 else F3D)] + list(s.seismograms()[:ndim])
        return out, s.energy() if energy else None


@pytest.mark.parametrize("order", [2, 4, 8])
@pytest.mark.parametrize("prec", [4, 8])
def test_2d_tiles_and_energy(order, prec):
    n, tol = (131, 150), (1e-12 if prec == 8 else 1e-4)
    base, en = _run(n, order, prec, True, 4)
    for tile in (4, 8, 16, 32, 64):
        for energy in (False, True):
            out, e = _run(n, order, prec, energy, tile)
            for a, b in zip(out, base):
                np.testing.assert_array_equal(a, b)
            for a, b in zip(e or (), en):
                assert rel_l2(a, b) <= tol
    assert np.abs(base[0]).max() > 0 and en[0].min() > 0


@pytest.mark.parametrize("prec", [4, 8])
def test_3d_tiles_chunks_and_energy(prec):
    n, tol = (70, 41, 37), (1e-12 if prec == 8 else 1e-4)
    base, en = _run(n, 2, prec, True, 4)
    for tile, kchunk in ((4, 1), (4, 16), (8, 3), (16, 0)):
        for energy in (False, True):
            out, e = _run(n, 2, prec, energy, tile, kchunk)
            for a, b in zip(out, base):
                np.testing.assert_array_equal(a, b)
            for a, b in zip(e or (), en):
                assert rel_l2(a, b) <= tol
