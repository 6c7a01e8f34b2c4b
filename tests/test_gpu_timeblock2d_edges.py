"""Time-blocked 2D step on grids whose axes have no absorbing slab, or slabs on
one side only, and grids narrower or lower than one strip or chunk: the split
of a grid's items into those with and without C-PML code per axis.  Energy and
receivers of a level that the next launch, or the end of the run, finishes.

Bar: bit-exact against the single-step kernels (fields, memory variables,
seismograms); energy 1e-12 (double) / 1e-4 (float) rel-L2, which sums the same
terms in another order.
"""
import numpy as np
import pytest

from gpu_runner import F2D, MEM2D, rel_l2
from seismic_cpml_amd import CpmlGpu, no_absorption
from seismic_cpml_amd import solver as S

pytestmark = pytest.mark.gpu


def _profile(n, kind, prec, dt):
    p = S.pml_profile(n, 10.0, dt, 6, 3300.0, 12.0, prec, use_min=kind in ("both", "min"),
                      use_max=kind in ("both", "max"))
    return no_absorption(n, prec) if kind == "none" else p


def _run(n, kinds, order, prec, tb, cadence, chunks):
    nx, ny = n
    dt = 0.4 * 10.0 / (3300.0 * 2 ** 0.5)
    nstep = chunks[-1][1]
    rng = np.random.default_rng(nx + ny)
    real = np.float32 if prec == 4 else np.float64
    with CpmlGpu(2, order, prec, nx, ny, 1, 10.0, 10.0, 1.0, dt, 6, nstep) as s:
        rho = rng.uniform(2000, 2600, (ny, nx)).astype(real)
        mu = (rho * 1900.0 ** 2).astype(real)
        s.set_medium((rho * 1.0e6).astype(real) + mu, mu, rho)
        s.set_pml(*(_profile(m, k, prec, dt) for m, k in zip(n, kinds)))
        f = np.sin(np.arange(nstep)).astype(real)
        s.set_source(nx // 2, ny // 3, 1, f, -f)
        s.set_receivers([2, nx // 2, nx - 1], [2, ny // 2, ny - 1])
        if cadence:
            s.set_energy(cadence)
        for name in ("vx", "vy"):
            v = np.zeros((ny, nx), real)
            v[2:-2, 2:-2] = rng.standard_normal((ny - 4, nx - 4))
            s.set_field(name, v)
        if tb:
            s.set_time_block(*tb)
        for a, b in chunks:
            s.run(a, b)
        out = {k: s.field(k) for k in F2D}
        out.update({"m_" + k: s.memory(k) for k in MEM2D})
        out.update(zip(("sisvx", "sisvy"), s.seismograms()))
        energy = s.energy() if cadence else None
    return out, energy


@pytest.mark.parametrize("n,kinds,order,tb,cadence", [
    ((300, 90), ("none", "none"), 2, (2, 0, 0), 1),
    ((131, 200), ("none", "both"), 4, (2, 0, 9), 3),
    ((257, 61), ("both", "none"), 4, (2, 17, 0), 0),
    ((150, 145), ("min", "max"), 2, (2, 56, 31), 2),
    ((120, 131), ("max", "min"), 8, (1, 0, 0), 1),
    ((23, 400), ("both", "both"), 4, (1, 0, 64), 0),
    ((400, 21), ("both", "min"), 2, (2, 0, 1), 1),
])
@pytest.mark.parametrize("prec", [4, 8])
def test_tb2d_axes_without_slabs_match_single_steps(n, kinds, order, tb, cadence, prec):
    chunks = [(1, 4), (5, 23), (24, 24), (25, 41)]
    a, ea = _run(n, kinds, order, prec, None, cadence, chunks)
    b, eb = _run(n, kinds, order, prec, tb, cadence, chunks)
    for k in a:
        np.testing.assert_array_equal(a[k], b[k], err_msg=k)
    assert np.abs(a["vx"]).max() > 0
    for p, q in zip(ea or (), eb or ()):
        assert rel_l2(q, p) <= (1e-12 if prec == 8 else 1e-4)
