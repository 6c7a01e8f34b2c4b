"""Time blocks in strips narrower than the lanes allow, on grids whose rows fill
whole cache lines: the lanes past a strip's ring lie beyond the grid while the
strip itself needs no x code, and the memory variables of the y and z slabs have
no ghost column for them to read.

Bar: bit-exact against the single-step kernels (2D, 3D), against the same shots
in single steps (batch).
"""
import numpy as np
import pytest

import test_gpu_timeblock2d_edges as edges2
import test_gpu_timeblock3d_edges as edges3
from seismic_cpml_amd import CpmlBatch, no_absorption
from seismic_cpml_amd import solver as S

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,kinds,order,tb", [
    ((256, 90), ("max", "both"), 2, (2, 40, 0)),
    ((256, 131), ("none", "both"), 4, (2, 31, 0)),
    ((128, 70), ("both", "max"), 2, (1, 9, 13)),
    ((320, 60), ("max", "both"), 8, (1, 24, 0)),
])
@pytest.mark.parametrize("prec", [4, 8])
def test_tb2d_narrow_strips(n, kinds, order, tb, prec):
    chunks = [(1, 17), (18, 40)]
    a, _ = edges2._run(n, kinds, order, prec, None, 0, chunks)
    b, _ = edges2._run(n, kinds, order, prec, tb, 0, chunks)
    for k in a:
        np.testing.assert_array_equal(a[k], b[k], err_msg=k)
    assert np.abs(a["vx"]).max() > 0


@pytest.mark.parametrize("n,kinds,tb", [
    ((128, 40, 33), ("max", "both", "both"), (2, 20, 7)),
    ((192, 31, 30), ("none", "both", "both"), (2, 37, 0)),
    ((64, 45, 40), ("none", "none", "both"), (1, 5, 9)),
])
@pytest.mark.parametrize("prec", [4, 8])
def test_tb3d_narrow_strips(n, kinds, tb, prec):
    a, b = edges3._run(n, kinds, prec, None), edges3._run(n, kinds, prec, tb)
    for k in a:
        np.testing.assert_array_equal(a[k], b[k], err_msg=k)
    assert np.abs(a["vx"]).max() > 0


@pytest.mark.parametrize("ow", [9, 23, 33])
@pytest.mark.parametrize("prec", [4, 8])
def test_batch_narrow_strips(ow, prec):
    real = np.float32 if prec == 4 else np.float64
    dt, nstep, order = 0.4 * 10.0 / (3300.0 * 2 ** 0.5), 31, 4
    grids = [(256, 64), (128, 100), (64, 80)]
    shots = [dict(NX=nx, NY=ny, DELTAX=10.0, DELTAY=10.0, DELTAT=dt, NPOINTS_PML=6)
             for nx, ny in grids]
    out = []
    for tb in (0, 2):
        with CpmlBatch(order, prec, shots, nstep) as b:
            rng = np.random.default_rng(5)
            for q, (nx, ny) in enumerate(grids):
                rho = rng.uniform(2000, 2600, (ny, nx)).astype(real)
                mu = (rho * 1900.0 ** 2).astype(real)
                b.set_medium(q, (rho * 1.0e6).astype(real) + mu, mu, rho)
                b.set_pml(q, no_absorption(nx, prec),
                          S.pml_profile(ny, 10.0, dt, 6, 3300.0, 12.0, prec))
                f = np.sin(np.arange(nstep)).astype(real)
                b.set_source(q, nx // 2, ny - 4, f, -f)
                b.set_receivers(q, [2, nx - 1], [3, ny - 2])
            if tb:
                b.set_time_block(tb, ow, 0)
            b.run()
            out.append([[b.field(q, k) for k in edges2.F2D] + list(b.seismograms(q))
                        for q in range(len(grids))])
    for p, r in zip(*out):
        for x, y in zip(p, r):
            np.testing.assert_array_equal(x, y)
        assert np.abs(p[0]).max() > 0
