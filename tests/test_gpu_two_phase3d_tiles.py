"""Two-phase 3D kernels (orders 2 and 4): tile heights, chunk depths and row
lengths at the edges of the tiles.  A column's values do not depend on the tile
that computes it.

Bar: bit-exact against 4-row tiles with one plane per chunk, where no plane's
values are loaded ahead; the default chunk depth (0 in the list) too."""
import numpy as np
import pytest

from gpu_runner import F3D, MEM3D
from seismic_cpml_amd import CpmlGpu
from seismic_cpml_amd import solver as S

pytestmark = pytest.mark.gpu


def _run(order, prec, n, tile, kchunk, nstep=9):
    nx, ny, nz = n
    dt = 0.4 * 10.0 / (4000.0 * 3 ** 0.5)
    rng = np.random.default_rng(sum(n))
    real = np.float32 if prec == 4 else np.float64
    with CpmlGpu(3, order, prec, nx, ny, nz, 10.0, 10.0, 10.0, dt, 5, nstep) as s:
        rho = rng.uniform(2000, 2600, (nz, ny, nx)).astype(real)
        mu = (rho * 2000.0 ** 2).astype(real)
        s.set_medium((rho * 2.0 * 2000.0 ** 2).astype(real), mu, rho)
        s.set_pml(*(S.pml_profile(m, 10.0, dt, 5, 4000.0, 12.0, prec) for m in n))
        f = np.sin(np.arange(nstep)).astype(real)
        s.set_source(nx // 2, ny // 3, nz // 2, f, -f)
        s.set_receivers([1, nx // 2, nx], [1, ny // 2, ny], [1, nz // 2, nz])
        for name in ("vx", "vy", "vz"):
            v = np.zeros((nz, ny, nx), real)
            v[2:-2, 2:-2, 2:-2] = rng.standard_normal((nz - 4, ny - 4, nx - 4))
            s.set_field(name, v)
        s.set_tile(tile)
        if kchunk:
            s.set_kchunk(kchunk)
        s.run()
        out = {k: s.field(k) for k in F3D}
        out.update({"m_" + k: s.memory(k) for k in MEM3D})
        out.update(zip(("sisvx", "sisvy", "sisvz"), s.seismograms()))
    return out


@pytest.mark.parametrize("order", [2, 4])
@pytest.mark.parametrize("prec", [4, 8])
@pytest.mark.parametrize("n", [(63, 17, 20), (64, 16, 33), (65, 31, 21), (129, 24, 16),
                               (21, 40, 29)])
def test_tiles_and_chunks_agree(order, prec, n):
    a = _run(order, prec, n, 4, 1)
    assert np.abs(a["vx"]).max() > 0
    for tile, kchunk in [(4, 0), (8, 7), (16, 2), (4, 64)]:
        b = _run(order, prec, n, tile, kchunk)
        for k in a:
            np.testing.assert_array_equal(a[k], b[k], err_msg=f"{tile} {kchunk} {k}")
