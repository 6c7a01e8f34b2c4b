"""Time-blocked 3D step on grids whose axes have no absorbing slab, or slabs
on one side only: the slab-free class of an axis holds the tiles strictly
inside the grid, so without a slab the tiles at the rigid faces must still go
to the class with that axis' predicates.  Also strips that store whole
64-byte sectors against strips that do not, and rows shorter than a tile.

Bar: bit-exact against the single-step kernels (fields, memory variables,
seismograms).
"""
import numpy as np
import pytest

from gpu_runner import F3D, MEM3D
from seismic_cpml_amd import CpmlGpu, no_absorption
from seismic_cpml_amd import solver as S

pytestmark = pytest.mark.gpu


def _profile(n, kind, prec, dt):
    p = S.pml_profile(n, 10.0, dt, 6, 4000.0, 12.0, prec, use_min=kind in ("both", "min"),
                      use_max=kind in ("both", "max"))
    return no_absorption(n, prec) if kind == "none" else p


def _run(n, kinds, prec, tb, nstep=23):
    nx, ny, nz = n
    dt = 0.5 * 10.0 / (4000.0 * 3 ** 0.5)
    rng = np.random.default_rng(sum(n))
    real = np.float32 if prec == 4 else np.float64
    with CpmlGpu(3, 2, prec, nx, ny, nz, 10.0, 10.0, 10.0, dt, 6, nstep) as s:
        shp = (nz, ny, nx)
        rho = rng.uniform(2000, 2600, shp).astype(real)
        mu = (rho * 2000.0 ** 2).astype(real)
        s.set_medium((rho * 2.0 * 2000.0 ** 2).astype(real), mu, rho)
        s.set_pml(*(_profile(m, k, prec, dt) for m, k in zip(n, kinds)))
        f = np.sin(np.arange(nstep)).astype(real)
        s.set_source(nx // 2, ny // 3, nz // 2, f, -f)
        s.set_receivers([1, nx // 2, nx], [1, ny // 2, ny], [1, nz // 2, nz])
        for q, name in enumerate(("vx", "vy", "vz")):
            v = rng.standard_normal(shp).astype(real)
            v[0] = v[-1] = v[:, 0] = v[:, -1] = v[:, :, 0] = v[:, :, -1] = 0
            s.set_field(name, v)
        if tb:
            s.set_time_block(*tb)
        s.run()
        out = {k: s.field(k) for k in F3D}
        out.update({"m_" + k: s.memory(k) for k in MEM3D})
        out.update(zip(("sisvx", "sisvy", "sisvz"), s.seismograms()))
    return out


@pytest.mark.parametrize("n,kinds,tb", [
    ((70, 40, 33), ("none", "none", "none"), (2, 0, 0)),
    ((131, 29, 30), ("none", "both", "both"), (2, 48, 7)),
    ((65, 64, 47), ("both", "none", "max"), (2, 56, 0)),
    ((150, 45, 40), ("min", "max", "none"), (2, 32, 11)),
    ((100, 31, 29), ("max", "min", "min"), (1, 0, 9)),
])
@pytest.mark.parametrize("prec", [4, 8])
def test_tb3d_axes_without_slabs_match_single_steps(n, kinds, tb, prec):
    a, b = _run(n, kinds, prec, None), _run(n, kinds, prec, tb)
    for k in a:
        np.testing.assert_array_equal(a[k], b[k], err_msg=k)
    assert np.abs(a["vx"]).max() > 0
