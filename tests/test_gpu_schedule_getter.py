"""GPU: the update order of the last sweep is read without changing the job: from several
threads at once, in part, and again later."""
import ctypes as C
import threading

import numpy as np
import pytest

from mbirtem import capi
from mbirtem import phantom as P

pytestmark = pytest.mark.gpu


def _job(ctx, n_r, n_t, n_z, views, **kw):
    ang = P.tilt_series(views, 60.0)
    geom = capi.geometry_init(n_r, n_t, ang, n_z / 2)
    y = np.random.default_rng(n_r).random((views, n_r, n_t), dtype=np.float32)
    return capi.Job(ctx, geom, ang, y, seed=5, **kw)


@pytest.mark.parametrize("n_r,n_t,n_z,kw", [
    (300, 9, 40, {}), (300, 65, 24, {}), (40, 9, 8, dict(kernel_mode=3)),
    (90, 5, 9, dict(schedule=1, rows_per_step=2)),
])
def test_concurrent_readers_see_the_sweep(gpu_ctx, n_r, n_t, n_z, kw):
    job = _job(gpu_ctx, n_r, n_t, n_z, 9, **kw)
    for it in range(2):
        job.sweep(0, it)
        got = [None] * 4

        def read(i):
            got[i] = [job.schedule() for _ in range(5)]

        th = [threading.Thread(target=read, args=(i,)) for i in range(4)]
        for t in th:
            t.start()
        for t in th:
            t.join()
        want = job.schedule()
        units = np.concatenate(want)
        assert len(np.unique(units[:, :2], axis=0)) == len(units) > 0
        for s in got:
            for steps in s:
                assert len(steps) == len(want)
                for a, b in zip(steps, want):
                    np.testing.assert_array_equal(a, b)
    job.close()


@pytest.mark.parametrize("cap", [0, 1, 257, 10 ** 6])
def test_part_of_the_units(gpu_ctx, cap):
    job = _job(gpu_ctx, 300, 9, 6, 9)
    job.sweep(0, 0)
    want = np.concatenate(job.schedule())
    out = np.full((len(want) + 1, 3), -7, np.int32)
    capi.lib().mbir_job_get_schedule(job.h, None, 0, out.ctypes.data_as(C.POINTER(C.c_int32)),
                                     min(cap, len(want)))
    n = min(cap, len(want))
    np.testing.assert_array_equal(out[:n], want[:n])
    assert (out[n:] == -7).all()
    job.close()
