"""Energy curves of grids with more tiles than the groups that their partial sums
are added in: a step whose sum is formed beside the next stress launch, and one
whose groups a launch of their own adds (the last step of a call or a graph, time
blocks).

Bars: the curve bit-exact however the run is cut, and with time blocks; 1e-12
(double) / 1e-4 (float) rel-L2 against the sum over the fields read back.
"""
import numpy as np
import pytest

from gpu_runner import rel_l2
from seismic_cpml_amd import CpmlGpu
from seismic_cpml_amd import solver as S
from test_gpu_step_finish import NSTEP, _energy, _run

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,order,window,tile", [
    ((700, 1000), 2, (6, 695, 6, 995), 4),              # 2750 tiles
    ((64, 8200), 4, (1, 64, 1, 8200), 4),               # 2050
    ((130, 200, 130), 2, (6, 125, 6, 195, 6, 125), 4),  # 2550, 8 planes each
])
@pytest.mark.parametrize("prec", [4, 8])
def test_many_tiles(n, order, window, tile, prec):
    ones = [(t, t) for t in range(1, NSTEP + 1)]
    states, _, en, medium = _run(n, order, prec, ones, window, 1, 0, tile)
    want = np.array([_energy(f, medium, window, len(n)) for f in states]).T
    for got, w in zip(en, want):
        assert rel_l2(got, w) <= (1e-12 if prec == 8 else 1e-4)
    for chunks, graph in (([(1, NSTEP)], 4), ([(1, NSTEP)], 0), ([(1, 5), (6, NSTEP)], 3)):
        for a, b in zip(_run(n, order, prec, chunks, window, 1, graph, tile)[2], en):
            np.testing.assert_array_equal(a, b)


@pytest.mark.parametrize("prec", [4, 8])
def test_many_tiles_time_blocked(prec):
    n = (130, 200, 130)
    dt = 0.4 * 10.0 / (4000.0 * 3 ** 0.5)
    real = np.float32 if prec == 4 else np.float64
    out = []
    for tb in (0, 2):
        rng = np.random.default_rng(11)
        with CpmlGpu(3, 2, prec, *n, 10.0, 10.0, 10.0, dt, 5, NSTEP) as s:
            rho = rng.uniform(2000, 2600, n[::-1]).astype(real)
            mu = (rho * 2000.0 ** 2).astype(real)
            s.set_medium((mu * 2).astype(real), mu, rho)
            s.set_pml(*(S.pml_profile(m, 10.0, dt, 5, 4000.0, 12.0, prec) for m in n))
            v = np.zeros(n[::-1], real)
            v[2:-2, 2:-2, 2:-2] = rng.standard_normal([m - 4 for m in n[::-1]])
            s.set_field("vx", v)
            s.set_energy(2)
            if tb:
                s.set_time_block(tb)
            s.run()
            out.append(s.energy())
    for a, b in zip(*out):
        np.testing.assert_array_equal(a, b)
        assert a[1::2].min() > 0
