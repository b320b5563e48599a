"""icon_mask3_filter over the widths it takes: the smallest and the largest,
odd and even, one and several slices, each side of the transform lengths
(2N - 1 against 128, 256, ..., 2048) and powers of two with and without the
chirp transform.  A random half-spectrum multiplier exercises every column,
kx = 0 and kx = N/2 (their masks' even parts) among them.

Tolerance: single-precision transforms of up to 2 x 4 lengths of 2048, each
with an rms error of ~1e-7 of the rms output; over up to 4e6 values the largest
is ~6 times the rms error, and the largest output is larger still: 2e-5 of the
largest output, the bound the other widths' tests use.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,count", [(8, 5), (9, 3), (33, 2), (64, 3), (65, 1), (101, 3), (128, 1), (129, 2), (256, 3),
                                     (465, 2), (512, 2), (513, 1), (1000, 1), (1023, 1), (1024, 2), (2048, 1)])
def test_mask3_filter_widths(icon, N, count):
    from oracle import mask3_ref
    print("mask3 filter N=%d, %d slices" % (N, count), flush=True)
    rng = np.random.default_rng(N)
    sl = rng.standard_normal((count, N, N)).astype(np.float32)
    half = rng.uniform(0, 2, (N, N // 2 + 1)).astype(np.float32)
    got, want = icon.icon.mask3_filter(sl, half), mask3_ref.filter_slices(sl, half)
    err = float(np.abs(got - want).max() / np.abs(want).max())
    print("  largest error %.1e" % err, flush=True)
    assert err <= 2e-5
