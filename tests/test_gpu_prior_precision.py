"""GPU: the prior sum's pair terms keep their FP64 bits: one voxel in an empty volume, whose
26 pairs have the same difference, so that a pair's error is not averaged away."""
import numpy as np
import pytest

from mbirtem import capi

pytestmark = pytest.mark.gpu

# u = 2^-53.  A pair: the square is exact, division 1 u; the power 2 u, its division and sum 1 u
# each; quotient 1 u, weight 1 u: 7 u.  The sum: 12 additions of the voxel's own 13 terms, then
# at most 26 more with the neighbours' (all others add exact zeros): 45 u in all.
TOL = 45 * 2.0 ** -53


@pytest.mark.parametrize("q,c,lo,hi", [(1.2, 1e-3, -9, 0), (1.05, 1e-60, -37, -33),
                                       (1.7, 1e-60, -37, -20), (1.0, 1e-3, -12, 3),
                                       (2.0, 1e-3, -9, 0)])
def test_pair_terms(gpu_ctx, q, c, lo, hi):
    n_r, n_t, n_z, sx = 16, 9, 6, 0.1
    ang = np.linspace(-60, 60, 5)
    geom = capi.geometry_init(n_r, n_t, ang, n_z / 2)
    job = capi.Job(gpu_ctx, geom, ang, np.zeros((5, n_r, n_t), np.float32), sigma_x=sx, mrf_q=q,
                   mrf_c=c)
    rng = np.random.default_rng(1)
    vol = np.zeros(job.vshape, np.float32)
    weights = np.longdouble(6 * 523 + 12 * 370 + 8 * 302) / 10000
    worst = 0.0
    for d in (10.0 ** rng.uniform(lo, hi, 40)).astype(np.float32):
        vol[2, 7, 4] = d
        job.set_volume(vol)
        got = job.cost(terms=True)[1][1]
        a = np.longdouble(d)
        t = np.power(a, np.longdouble(2.0 - q)) / np.longdouble(sx ** (2.0 - q))
        want = weights * (a * a / np.longdouble(sx ** 2.0)) / (np.longdouble(c) + t)
        worst = max(worst, abs(float((got - want) / want)))
    job.close()
    assert worst <= TOL
