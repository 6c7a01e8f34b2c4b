"""set_field / field through the pinned staging buffers: one and several
buffers' worth, an odd number of buffers, rows that do not fill a wavefront, and
arrays that the caller has pinned.

Bar: the values come back bit for bit, and other fields keep theirs."""
import numpy as np
import pytest
import torch

from seismic_cpml_amd import CpmlGpu

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ndim,order,n", [(2, 2, (61, 50, 1)), (2, 4, (1301, 1403, 1)),
                                          (2, 8, (4000, 1100, 1)), (3, 2, (96, 80, 72)),
                                          (3, 2, (30, 257, 300)), (3, 4, (191, 203, 131)),
                                          (3, 2, (640, 610, 45))])
@pytest.mark.parametrize("prec", [4, 8])
def test_field_round_trip(ndim, order, n, prec):
    nx, ny, nz = n
    rng = np.random.default_rng(nx)
    real = np.float32 if prec == 4 else np.float64
    shape = (nz, ny, nx)[3 - ndim:]
    with CpmlGpu(ndim, order, prec, nx, ny, nz, 10.0, 10.0, 10.0, 1e-3, 6, 4) as s:
        a = {k: rng.standard_normal(shape).astype(real) for k in ("vx", "sigmaxy")}
        for k, v in a.items():
            s.set_field(k, v)
        pinned = torch.empty(shape, dtype=torch.float32 if prec == 4 else torch.float64,
                             pin_memory=True)
        a["sigmaxx"] = pinned.numpy()
        a["sigmaxx"][:] = a["vx"][::-1]
        s.set_field("sigmaxx", a["sigmaxx"])
        for k, v in a.items():
            np.testing.assert_array_equal(s.field(k), v)
        assert not s.field("vy").any()
