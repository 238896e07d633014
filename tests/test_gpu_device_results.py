"""GPU: results go to device memory as well as to host memory, below and above the size from
which host memory is filled through staging chunks."""
import ctypes as C

import numpy as np
import pytest

from mbirtem import capi

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n_r,n_t,n_z", [(16, 9, 6), (63, 64, 64), (64, 64, 64), (65, 64, 300)])
def test_results_into_device_memory(gpu_ctx, n_r, n_t, n_z):
    import torch
    ang = np.linspace(-60.0, 60.0, 5)
    geom = capi.geometry_init(n_r, n_t, ang, n_z / 2)
    job = capi.Job(gpu_ctx, geom, ang, np.zeros((5, n_r, n_t), np.float32))
    vol = np.random.default_rng(n_r).random(job.vshape, dtype=np.float32)
    job.set_volume(vol)
    out = torch.full(vol.shape, -1.0, device="cuda")
    torch.cuda.synchronize()
    assert capi.lib().mbir_job_get_volume(job.h, C.cast(out.data_ptr(), C.POINTER(C.c_float))) == 0
    np.testing.assert_array_equal(out.cpu().numpy(), vol)
    pinned = torch.empty(vol.shape, pin_memory=True)
    assert capi.lib().mbir_job_get_volume(job.h, C.cast(pinned.data_ptr(),
                                                        C.POINTER(C.c_float))) == 0
    np.testing.assert_array_equal(pinned.numpy(), vol)
    job.close()
