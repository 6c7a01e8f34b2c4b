"""Single steps whose receivers, energy sum and step counter the next stress
launch (or the end of the call) finishes, and whose velocity launch sums the
energy: runs cut into calls of one, two and many steps, graphs and eager
launches, tile heights, cadences and energy windows that cut tiles.

Bars: seismograms and fields bit-exact however the run is cut; the energy of
every step 1e-12 (double) / 1e-4 (float) rel-L2 against the sum over the fields
read back after that step."""
import numpy as np
import pytest

from gpu_runner import F2D, F3D, rel_l2
from seismic_cpml_amd import CpmlGpu
from seismic_cpml_amd import solver as S

pytestmark = pytest.mark.gpu

NSTEP = 12


def _run(n, order, prec, chunks, window, cadence, graph=4, tile=4):
    ndim = len(n)
    nx, ny, nz = (*n, 1)[:3]
    dt = 0.4 * 10.0 / (4000.0 * 3 ** 0.5)
    rng = np.random.default_rng(sum(n))
    real = np.float32 if prec == 4 else np.float64
    shape = n[::-1]
    with CpmlGpu(ndim, order, prec, nx, ny, nz, 10.0, 10.0, 10.0, dt, 5, NSTEP) as s:
        rho = rng.uniform(2000, 2600, shape).astype(real)
        mu = (rho * 2000.0 ** 2).astype(real)
        lam = (mu * 2).astype(real)
        s.set_medium(lam, mu, rho)
        s.set_pml(*(S.pml_profile(m, 10.0, dt, 5, 4000.0, 12.0, prec) for m in n))
        f = np.sin(np.arange(NSTEP)).astype(real)
        s.set_source(nx // 2, ny // 3, max(nz // 2, 1), f, -f)
        idx = [[1 + m // 3, m // 2] for m in n]
        s.set_receivers(*idx)
        for name in ("vx", "vy", "vz")[:ndim]:
            v = np.zeros(shape, real)
            v[(slice(2, -2),) * ndim] = rng.standard_normal([m - 4 for m in shape])
            s.set_field(name, v)
        s.set_energy(cadence, window)
        s.set_graph_steps(graph)
        s.set_tile(tile)
        states = []
        for a, b in chunks:
            s.run(a, b)
            states.append({k: s.field(k) for k in (F2D if ndim == 2 else F3D)})
        return states, s.seismograms()[:ndim], s.energy(), (lam, mu, rho)


def _energy(f, medium, window, ndim):
    cut = tuple(slice(window[2 * a] - 1, window[2 * a + 1]) for a in reversed(range(ndim)))
    f = {k: v[cut].astype(np.float64) for k, v in f.items()}
    l, m, r = (a[cut].astype(np.float64) for a in medium)
    v2 = sum(f[k] ** 2 for k in ("vx", "vy", "vz")[:ndim])
    if ndim == 2:
        x, y, q = f["sigmaxx"], f["sigmayy"], f["sigmaxy"]
        den = 4 * m * (l + m)
        pot = ((l + 2 * m) * x - l * y) / den * x + ((l + 2 * m) * y - l * x) / den * y \
            + q * q / m
    else:
        x, y, z = f["sigmaxx"], f["sigmayy"], f["sigmazz"]
        den = 2 * m * (3 * l + 2 * m)
        pot = (2 * (l + m) * x - l * y - l * z) / den * x \
            + 2 * (2 * (l + m) * y - l * x - l * z) / den * y \
            + sum(f[k] ** 2 for k in ("sigmaxy", "sigmaxz", "sigmayz")) / m
    return 0.5 * (r * v2).sum(), 0.5 * pot.sum()


@pytest.mark.parametrize("n,order,window,cadence,tile", [
    ((70, 61), 2, (6, 65, 6, 56), 1, 4),
    ((131, 40), 4, (1, 131, 1, 40), 1, 16),
    ((64, 70), 8, (9, 9, 3, 70), 2, 32),
    ((66, 30, 29), 2, (6, 61, 6, 25, 6, 24), 1, 4),
    ((40, 33, 27), 2, (1, 40, 2, 33, 27, 27), 3, 8),
    ((21, 20, 40), 4, (6, 16, 6, 15, 1, 40), 1, 4),
])
@pytest.mark.parametrize("prec", [4, 8])
def test_steps_finished_by_the_next(n, order, window, cadence, tile, prec):
    ones = [(t, t) for t in range(1, NSTEP + 1)]
    tol = 1e-12 if prec == 8 else 1e-4
    states, sis, en, medium = _run(n, order, prec, ones, window, cadence, 0, tile)
    want = np.array([_energy(f, medium, window, len(n)) if (t + 1) % cadence == 0 else (0, 0)
                     for t, f in enumerate(states)]).T
    for got, w in zip(en, want):
        assert rel_l2(got, w) <= tol
    for chunks, graph in (([(1, NSTEP)], 4), ([(1, NSTEP)], 0), ([(1, 2), (3, 9), (10, NSTEP)], 3)):
        st, si, e2, _ = _run(n, order, prec, chunks, window, cadence, graph, tile)
        for k, v in st[-1].items():
            np.testing.assert_array_equal(v, states[-1][k], err_msg=k)
        for a, b in zip(si, sis):
            np.testing.assert_array_equal(a, b)
        for a, b in zip(e2, en):
            np.testing.assert_array_equal(a, b)
