"""GPU: the bright-field line update's short root, quotient and selector against the general
root, division and comparison, on the device and bit for bit."""
import ctypes as C

import pytest

import native_checks

pytestmark = pytest.mark.gpu


# (what, comparisons per thread of 2^19, at least so many in all)
@pytest.mark.parametrize("name,what,per,least", [
    ("root", 0, 0, 99 * 2 ** 23),          # every float of the range
    ("quotient", 1, 2048, 2 ** 29),        # 2^30 seeded pairs
    ("midpoint", 2, 0, 2 ** 24),           # quotients next to the middle of two floats
    ("factor", 3, 512, 2 ** 26),
    ("selector", 4, 512, 2 ** 26),
])
def test_short_forms_keep_the_bits(gpu_ctx, name, what, per, least):
    out = (C.c_ulonglong * 2)()
    assert native_checks.load().checks_selector(what, 12345, per, out) == 0
    assert out[0] >= least
    assert out[1] == 0, f"{out[1]} of {out[0]} differ"
