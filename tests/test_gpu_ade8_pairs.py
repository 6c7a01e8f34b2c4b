"""ADE-PML RK4 step with two stages per pass away from the PML band: box sizes
at the edges of strips and chunks, the source inside the box, in the frame and
where they meet.  A band wide enough to cover the grid leaves every stage a pass
of its own; with absorbing coefficients only in the outer points (0 and K = 1
elsewhere) both compute the same.

Bar: bit-exact fields and seismograms."""
import numpy as np
import pytest

from seismic_cpml_amd import CpmlGpu, no_absorption
from seismic_cpml_amd import solver as S

pytestmark = pytest.mark.gpu

NSTEP = 13
NAMES = ("vx", "vy", "sigmaxx", "sigmayy", "sigmaxy")


def _run(n, npml, width, prec, src):
    nx, ny = n
    rng = np.random.default_rng(nx * ny)
    real = np.float32 if prec == 4 else np.float64
    dt = 5e-4
    prof = [S.pml_profile(m, 10.0, dt, width, 3300.0, 12.0, prec) if width
            else no_absorption(m, prec) for m in n]
    tables = {}
    for ax, p in zip("xy", prof):
        for q, k in ((0, "a_"), (1, "b_"), (3, "ah_"), (4, "bh_")):
            scale = np.array([1.0, 0.9, 0.8, 0.7])[:, None]
            tables[k + ax] = (np.asarray(p[q])[None] * scale).astype(real)
    f = rng.standard_normal((NSTEP, 4)).astype(real)
    with CpmlGpu(2, 8, prec, nx, ny, 1, 10.0, 9.0, 1.0, dt, npml, NSTEP) as s:
        rho = rng.uniform(2000, 2600, (ny, nx)).astype(real)
        mu = (rho * 1900.0 ** 2).astype(real)
        s.set_medium((mu * 1.3).astype(real), mu, rho)
        s.set_pml(*prof)
        s.set_ade_rk4(tables, 1e3 * f, -1e3 * f)
        s.set_source(*src, 1, np.zeros(NSTEP, real), np.zeros(NSTEP, real))
        s.set_receivers([20, nx // 2, nx - 18], [20, ny // 2, ny - 18])
        for k in NAMES:
            s.set_field(k, (rng.standard_normal((ny, nx)) * (1 if k[0] == "v" else 1e6)).astype(real))
        s.run(1, 5)
        s.run(6, NSTEP)
        out = {k: s.field(k) for k in NAMES}
        out.update(zip(("sisvx", "sisvy"), s.seismograms()))
    return out


@pytest.mark.parametrize("n,width,src", [
    ((1130, 1120), 6, (50, 50)),
    ((6100, 270), 10, (18, 30)),     # the source beside the box
    ((281, 6003), 0, (32, 13)),      # no band: the box starts off the edges
    ((1301, 1029), 10, (64, 96)),
    ((2200, 753), 20, (200, 137)),
])
@pytest.mark.parametrize("prec", [4, 8])
def test_pairs_of_stages_match_single_stages(n, width, src, prec):
    a = _run(n, (min(n) - 8) // 2, width, prec, src)
    b = _run(n, width, width, prec, src)
    for k in a:
        np.testing.assert_array_equal(a[k], b[k], err_msg=k)
    assert np.isfinite(a["vx"]).all() and np.abs(a["sisvx"]).max() > 0
