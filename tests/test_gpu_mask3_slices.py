"""icon_mask3_filter: a slice's result is its own.  Stacks of odd and even
widths whose slices differ by six orders of magnitude, and whose first slice
ends in a NaN and an infinity: every other slice must have the bits that it has
when it is filtered alone.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N", [9, 33, 63, 64, 101, 128, 200, 465, 1023])
def test_mask3_slices_are_independent(icon, N):
    print("mask3 slices alone and in a stack, N=%d" % N, flush=True)
    rng = np.random.default_rng(N)
    sl = rng.standard_normal((4, N, N)).astype(np.float32)
    sl[0, -1, 3] = np.nan
    sl[0, -1, 4] = np.inf
    sl[2] *= np.float32(1e6)
    half = rng.uniform(0, 2, (N, N // 2 + 1)).astype(np.float32)
    stack = icon.icon.mask3_filter(sl, half)
    for k in (1, 2, 3):
        np.testing.assert_array_equal(stack[k], icon.icon.mask3_filter(sl[k:k + 1], half)[0])
