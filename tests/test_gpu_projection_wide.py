"""GPU: the projection's form for volumes of 2^30 voxels and more (64-bit line addresses), at
small sizes against the ordinary form, which is checked against the oracle: the same entries
in the same order, so the same bits."""
import ctypes as C

import numpy as np
import pytest

import native_checks
from mbirtem import capi

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n_r,n_t,n_z,ratio,angles", [
    (3, 1, 2, 1, (-60.0, 0.0, 60.0)),                                # one slice
    (33, 7, 18, 1, (-72.0, -45.0, -10.0, 0.0, 45.0, 72.0)),          # lanes shared by 8 lines
    (34, 9, 8, 1, (-90.0, -80.0, 80.0, 90.0)), (37, 64, 10, 1, (-65.0, 3.0, 65.0)),
    (20, 65, 6, 1, (-50.0, 50.0)), (20, 128, 6, 1, (-50.0, 50.0)),   # two slices per lane
    (18, 129, 4, 1, (-60.0, 60.0)), (16, 256, 4, 1, (30.0,)),        # four
    (40, 11, 16, 2, (-70.0, 0.0, 70.0)), (64, 16, 16, 4, (-60.0, 20.0)),
])
def test_wide_projection_keeps_the_bits(gpu_ctx, n_r, n_t, n_z, ratio, angles):
    ang = np.asarray(angles)
    geom = capi.geometry_init(n_r, n_t, ang, n_z / 2, delta_xz_in=float(ratio),
                              interpolate_factor=float(ratio))
    rng = np.random.default_rng(n_r * 1000 + n_t)
    gains = rng.uniform(0.8, 1.2, len(ang))
    gains *= len(ang) / gains.sum()
    job = capi.Job(gpu_ctx, geom, ang, np.zeros((len(ang), n_r, n_t), np.float32), init_gain=gains)
    vol = rng.uniform(0.1, 1.0, job.vshape).astype(np.float32)
    vol[rng.uniform(size=vol.shape) < 0.3] = 0.0
    want = job.forward_project(vol)
    got = np.full(want.shape, np.nan)
    assert native_checks.load().checks_project_wide(
        job.h, vol.ctypes.data_as(C.POINTER(C.c_float)), got.ctypes.data_as(C.POINTER(C.c_double))) == 0
    job.close()
    assert want.max() > 0
    np.testing.assert_array_equal(got, want)
