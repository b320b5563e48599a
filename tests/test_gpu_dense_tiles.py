"""The solve with few slices (the dense tiles' interpolation entries shared
among further blocks, the grid in the other half of its buffer) against the same
slices in a batch that is too large for that: the two paths do the same
arithmetic, so results and residuals are equal to the last bit.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,depth,step,big", [(64, 64, 6, 600), (256, 256, 2, 40), (200, 120, 3, 70), (512, 300, 1, 20)])
def test_few_slices_equal_many(icon, N, depth, step, big):
    from feilab_amd.icon import Plan
    print("dense tiles", N, depth, step, big, flush=True)
    tilt = np.arange(-60, 60.1, step).astype(np.float32)
    rng = np.random.default_rng(N)
    sino = rng.standard_normal((big, len(tilt), N)).astype(np.float32)
    plan = Plan(N, tilt, thickness=depth, max_slices=big, device=0)
    few, rf, _ = plan.solve(sino[:1], 2, 9, 2, 2, 0.0, trace=True)
    many, rm, _ = plan.solve(sino, 2, 9, 2, 2, 0.0, trace=True)
    np.testing.assert_array_equal(few[0], many[0])
    np.testing.assert_array_equal(np.asarray(rf).reshape(1, -1)[0], np.asarray(rm).reshape(big, -1)[0])
