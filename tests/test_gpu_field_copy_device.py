"""Field arrays of the caller that lie in device memory: the host must not touch
them, so they don't go through the staging buffers.

Bar: the values come back bit for bit.
"""
import ctypes as C

import numpy as np
import pytest
import torch

from seismic_cpml_amd import CpmlGpu
from seismic_cpml_amd.solver import FIELDS

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ndim,n", [(2, (131, 90, 1)), (3, (40, 33, 21))])
@pytest.mark.parametrize("prec", [4, 8])
def test_device_arrays(ndim, n, prec):
    nx, ny, nz = n
    shape = (nz, ny, nx)[3 - ndim:]
    a = torch.randn(shape, dtype=torch.float32 if prec == 4 else torch.float64, device="cuda")
    b = torch.zeros_like(a)
    torch.cuda.synchronize()
    with CpmlGpu(ndim, 2, prec, nx, ny, nz, 10.0, 10.0, 10.0, 1e-3, 6, 4) as s:
        q = FIELDS.index("sigmaxy")
        s._call("cpml_gpu_set_field", q, C.c_void_p(a.data_ptr()))
        np.testing.assert_array_equal(s.field("sigmaxy"), a.cpu().numpy())
        s._call("cpml_gpu_get_field", q, C.c_void_p(b.data_ptr()))
    torch.cuda.synchronize()
    assert torch.equal(a, b)
