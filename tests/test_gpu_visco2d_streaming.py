"""2D viscoelastic step on a state larger than the caches, whose attenuation
memory variables stream past them, on ragged rows: every point of a window of
the large grid against the same window run as a small grid of its own (which
stays in the caches) where the window's edges cannot have reached it yet.

Bar: bit-exact (fields and attenuation memory variables).
"""
import numpy as np
import pytest

from gpu_runner import F2D
from seismic_cpml_amd import CpmlGpu, no_absorption

pytestmark = pytest.mark.gpu

NSTEP = 3
MARGIN = 4 * NSTEP  # a 4th-order step reaches 2 points in sigma and 2 more in v
TAUS = tuple(np.array([0.021, 0.004, 0.0009]) * k for k in (1.0, 0.92, 1.05, 0.9))


def _run(order, prec, lam, mu, rho, v):
    ny, nx = rho.shape
    with CpmlGpu(2, order, prec, nx, ny, 1, 10.0, 10.0, 1.0, 5e-4, 0, NSTEP) as s:
        s.set_medium(lam, mu, rho)
        s.set_pml(no_absorption(nx, prec), no_absorption(ny, prec))
        s.set_attenuation(*TAUS)
        for name, a in zip(("vx", "vy"), v):
            s.set_field(name, a)
        s.run()
        out = {k: s.field(k) for k in F2D}
        out.update({f"r{q}": s.attenuation_memory(q) for q in range(3)})
    return out


@pytest.mark.parametrize("order", [2, 4])
@pytest.mark.parametrize("prec,nx,ny", [(8, 1667, 1300), (4, 2501, 1700)])
def test_streaming_visco2d_matches_windows(order, prec, nx, ny):
    real = np.float32 if prec == 4 else np.float64
    rng = np.random.default_rng(3)
    rho = rng.uniform(2000, 2600, (ny, nx)).astype(real)
    mu = (rho * 1900.0 ** 2).astype(real)
    lam = (rho * 1.0e6).astype(real) + mu
    v = [rng.standard_normal((ny, nx)).astype(real) for _ in range(2)]
    for a in v:
        a[0] = a[-1] = a[:, 0] = a[:, -1] = 0
    big = _run(order, prec, lam, mu, rho, v)
    m = MARGIN
    for x, y in [(0, 0), (777, 401), (nx - 150, ny - 90), (64, ny - 90)]:
        w = np.s_[y:y + 90, x:x + 150]
        small = _run(order, prec, lam[w], mu[w], rho[w], [a[w] for a in v])
        # the window's own edges, but not those that are the grid's
        x0, x1 = (0 if x == 0 else m), (150 if x + 150 == nx else 150 - m)
        y0, y1 = (0 if y == 0 else m), (90 if y + 90 == ny else 90 - m)
        for k in small:
            np.testing.assert_array_equal(small[k][..., y0:y1, x0:x1],
                                          big[k][(..., *w)][..., y0:y1, x0:x1],
                                          err_msg=f"{k} {x} {y}")
            assert np.abs(small[k]).max() > 0
