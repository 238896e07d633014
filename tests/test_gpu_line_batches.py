"""GPU: the register-held line update at every batch that it is compiled for, in every launch
that takes it, against the batched kernel without prefetch, which walks every stream in loops:
the same bits.  The batch and the units of a step are worked out from the job and asserted,
so that a row cannot land on another form."""
import numpy as np
import pytest

from mbirtem import capi
from mbirtem import phantom as P
from test_gpu_line_forms import _run

pytestmark = pytest.mark.gpu

VIEWS = {8: 25, 12: 41, 16: 55, 20: 70, 24: 85, 28: 100, 32: 115, 36: 130, 40: 141}
SMALL, ARGS = 96, 256  # units in the launch's arguments (two sizes); more than 256: wide


def _data(n_r, n_t, views, bf, seed):
    rng = np.random.default_rng(seed)
    r = np.linspace(-1, 1, n_r)[None, :, None]
    base = np.maximum(0.0, 1 - 2 * r * r) * np.ones((views, n_r, n_t))
    if not bf:
        return (base + 0.03 * rng.standard_normal(base.shape)).astype(np.float32)
    y = 2000.0 * np.exp(-0.1 * base) + 45.0 * rng.standard_normal(base.shape)
    y[rng.uniform(size=y.shape) < 0.03] *= 0.3  # far below the model: rejected by the selector
    return np.maximum(y, 1.0).astype(np.float32)


def _batch_and_units(ctx, geom, ang, y):
    job = capi.Job(ctx, geom, ang, y)
    n = max(len(job.column(z, x)[0]) for z in range(geom.N_z) for x in range(geom.N_x))
    job.sweep(0, 0)
    steps = job.schedule()
    job.close()
    assert all((s[:, 2] == geom.N_y).all() for s in steps)  # whole lines
    units = [len(s) for s in steps]
    lanes = 1
    while lanes < min(geom.N_y, 64):
        lanes *= 2
    streams = 8 * (64 // lanes)
    return n, -(-(-(-n // streams)) // 4) * 4, max(units)


def _compare(ctx, n_r, n_t, n_z, views, bf, batch, lo, hi, entries=0):
    ang = P.tilt_series(views, 60.0)
    geom = capi.geometry_init(n_r, n_t, ang, n_z / 2)
    y = _data(n_r, n_t, views, bf, n_r + views)
    n, b, units = _batch_and_units(ctx, geom, ang, y)
    assert b == batch and lo < units <= hi and n > entries
    want = _run(ctx, geom, ang, y, 1, 0, bf, 0, 1.0)
    assert want[0].max() > 0
    for mode, prefetch in ((0, 0), (1, 1)):
        for a, c in zip(_run(ctx, geom, ang, y, mode, prefetch, bf, 0, 1.0), want):
            np.testing.assert_array_equal(a, c)


@pytest.mark.parametrize("bf", [0, 1])
@pytest.mark.parametrize("batch", sorted(VIEWS))
def test_units_in_the_arguments(gpu_ctx, batch, bf):
    _compare(gpu_ctx, 700, 33, 2, VIEWS[batch], bf, batch, SMALL, ARGS)


@pytest.mark.parametrize("bf", [0, 1])
@pytest.mark.parametrize("batch", sorted(VIEWS))
def test_few_units(gpu_ctx, batch, bf):
    _compare(gpu_ctx, 40, 64, 4, VIEWS[batch], bf, batch, 0, SMALL)


@pytest.mark.parametrize("bf", [0, 1])
@pytest.mark.parametrize("batch", sorted(VIEWS))
def test_wide_steps(gpu_ctx, batch, bf):
    _compare(gpu_ctx, 1500, 33, 2, VIEWS[batch], bf, batch, ARGS, 10 ** 6)


@pytest.mark.parametrize("bf", [0, 1])
@pytest.mark.parametrize("n_r,n_t,n_z,views,batch", [
    (24, 12, 8, 300, 20),   # lanes of 16 slices, 32 streams: a column of more than 512 entries
    (24, 30, 8, 300, 40),   # lanes of 32
])
def test_columns_of_more_entries_than_threads(gpu_ctx, n_r, n_t, n_z, views, batch, bf):
    _compare(gpu_ctx, n_r, n_t, n_z, views, bf, batch, 0, SMALL, entries=512)
