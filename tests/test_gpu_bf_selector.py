"""GPU: the Bragg selector that the line update leaves behind is |e sqrt(w)| < T in float32,
entry by entry, for every threshold that a problem may carry."""
import numpy as np
import pytest

from mbirtem import capi
from mbirtem import phantom as P

pytestmark = pytest.mark.gpu


# thresholds: ordinary ones, none above, not positive, with squares that are subnormal or
# overflow; counts whose weights are subnormal; lanes of 8 (general form), 32 and 64 slices,
# steps of more units than compute units
@pytest.mark.parametrize("mode", [0, 1])
@pytest.mark.parametrize("n_r,n_t,n_z,views,scale,T", [
    (24, 64, 8, 61, 1.0, 3.0), (24, 64, 8, 61, 1.0, 0.25), (24, 8, 8, 61, 1.0, 1.0),
    (24, 20, 8, 61, 1.0, -3.0), (24, 64, 8, 61, 1.0, 0.0), (24, 64, 8, 61, 1.0, 1e30),
    (24, 64, 8, 121, 5e-46, 1e-21), (24, 8, 8, 121, 5e-46, 1e-21),
    (24, 64, 8, 121, 5e-46, 3e-23), (24, 8, 8, 121, 5e-46, 3e-23), (24, 64, 8, 121, 5e-46, 1e-22),
    (1100, 33, 4, 41, 1.0, -0.5), (1100, 33, 4, 41, 1.0, 2.0),
])
def test_selector_is_the_comparison(gpu_ctx, n_r, n_t, n_z, views, scale, T, mode):
    ang = P.tilt_series(views, 60.0)
    geom = capi.geometry_init(n_r, n_t, ang, n_z / 2)
    rng = np.random.default_rng(n_t + views)
    counts = np.maximum(rng.poisson(2000.0 * np.exp(-0.2 * rng.random((views, n_r, n_t)))), 1)
    counts = (counts * scale).astype(np.float32)
    assert counts.min() > 0
    job = capi.Job(gpu_ctx, geom, ang, counts, bf_mode=1, bragg_T=T, seed=3, kernel_mode=mode,
                   sigma_x=0.002, mrf_c=0.01, default_offset=-np.log(2000.0 * scale),
                   default_variance=1.0, default_recon=0.0, noise_model=0)
    touched = job.forward_project(np.ones(job.vshape, np.float32)) > 0
    job.sweep(0, 0)  # no zero skipping yet: every slice refreshes its entries
    e, w, sel = job.error_sinogram(), job.weights(), job.selector()
    job.close()
    want = np.abs(e * np.sqrt(w)) < np.float32(T)
    assert touched.any()
    np.testing.assert_array_equal(sel.astype(bool)[touched], want[touched])
    assert sel[~touched].all()
