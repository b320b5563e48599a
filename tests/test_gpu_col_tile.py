"""The column tile (icon_plan_set_col_block) is a choice of the transforms'
kernels: solves keep their bits with either width, on every grid that has both.
"""
import numpy as np
import pytest

from feilab_amd import phantom

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,depth", [(64, 200), (200, 120), (256, 256), (500, 300), (512, 512)])
def test_solve_keeps_its_bits_with_either_tile(icon, N, depth):
    print("column tile 8 and 16, width %d, thickness %d" % (N, depth), flush=True)
    tilt = phantom.tilt_series(60, 5)
    sino = np.random.default_rng(N).standard_normal((2, len(tilt), N)).astype(np.float32)
    plan = icon.Plan(N, tilt, thickness=depth, max_slices=2)
    m8, r8, a8 = plan.solve(sino, 2, 9, 2, 2, 0.0, trace=True)
    for tile in (16, 8):
        plan.set_col_block(tile)
        assert plan.info.col_block == tile
        m, r, a = plan.solve(sino, 2, 9, 2, 2, 0.0, trace=True)
        np.testing.assert_array_equal(m, m8)
        np.testing.assert_array_equal(r, r8)
        np.testing.assert_array_equal(a, a8)
