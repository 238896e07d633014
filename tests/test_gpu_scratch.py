"""GPU: what a context keeps between calls is bounded, and a server's budget covers it."""
import numpy as np
import pytest

from mbirtem import capi

pytestmark = pytest.mark.gpu

KEEP = 64 << 20
SLACK = 8 << 20  # the driver's own granules


def _free():
    import torch
    torch.cuda.synchronize()
    return torch.cuda.mem_get_info(0)[0]


def _problem(views, n_r, n_t):
    ang = np.linspace(-60.0, 60.0, views)
    return capi.geometry_init(n_r, n_t, ang, 1.0), ang, np.zeros((views, n_r, n_t), np.float32)


@pytest.mark.parametrize("views,n_r,n_t,kept", [
    (64, 512, 128, True),     # 34 MB of scratch: kept for the next call
    (128, 512, 128, True),    # 64 MiB exactly
    (129, 512, 128, False),   # and more: given back at the end of the call
    (300, 1024, 128, False),
])
def test_kept_scratch_is_bounded(gpu_ctx, views, n_r, n_t, kept):
    ctx = capi.Context(0)
    capi.Job(ctx, *_problem(3, 16, 8)).close()
    before = _free()
    capi.Job(ctx, *_problem(views, n_r, n_t)).close()
    held = before - _free()
    ctx.close()
    assert held <= (KEEP if kept else 0) + SLACK
    assert before - _free() <= SLACK


def test_server_budget_covers_the_scratch(gpu_ctx):
    """The block of an earlier large call is given back once it no longer fits the budget,
    and kept where it does."""
    small = _problem(5, 24, 8)
    need = capi.problem_device_bytes(*small)
    for budget, kept in ((2 * need, False), (1 << 33, True)):
        ctx = capi.Context(0)
        srv = capi.Server(ctx, hbm_budget_bytes=budget, setup_threads=1)
        srv.wait(srv.submit(*small))
        before = _free()
        capi.Job(ctx, *_problem(100, 512, 128)).close()  # 52 MB of scratch
        assert before - _free() >= 48 << 20
        srv.wait(srv.submit(*small))
        srv.wait(srv.submit(*small))  # (the second setup begins behind the first one's end)
        held = before - _free()
        srv.close()
        ctx.close()
        assert (held >= 48 << 20) if kept else (held <= SLACK)


def test_scratch_given_back_and_made_again(gpu_ctx):
    """Projections before and after a call that is too large to keep, and of several sizes."""
    ctx = capi.Context(0)
    want = {}
    for views, n_r, n_t in [(5, 24, 8), (129, 512, 128), (5, 24, 8), (64, 512, 128), (129, 512, 128)]:
        job = capi.Job(ctx, *_problem(views, n_r, n_t))
        vol = np.random.default_rng(views).random(job.vshape, dtype=np.float32)
        got = job.forward_project(vol)
        job.close()
        np.testing.assert_array_equal(got, want.setdefault((views, n_r), got))
        assert got.max() > 0
    ctx.close()
