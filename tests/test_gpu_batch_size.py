"""A slice's images, residual trace and step sizes have the same bits whatever
the number of slices solved with it (more and fewer slices than compute units,
so that the residual's rows are shared among different numbers of blocks).
"""
import numpy as np
import pytest

from feilab_amd import phantom

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,depth,step", [(256, 64, 2), (200, 64, 2), (64, 64, 6), (300, 40, 1)])
def test_solve_does_not_depend_on_the_batch(icon, N, depth, step):
    S = 300
    print("1, 3 and %d slices, width %d, %d degrees" % (S, N, step), flush=True)
    tilt = phantom.tilt_series(60, step)
    sino = np.random.default_rng(N + step).standard_normal((S, len(tilt), N)).astype(np.float32)
    plan = icon.Plan(N, tilt, thickness=depth, max_slices=S)
    m, r, a = plan.solve(sino, 1, 3, 1, 2, 0.0, trace=True)
    r, a = np.asarray(r).reshape(S, -1), np.asarray(a).reshape(S, -1)
    for few in (1, 3, 70):
        mf, rf, af = plan.solve(sino[:few], 1, 3, 1, 2, 0.0, trace=True)
        np.testing.assert_array_equal(mf, m[:few])
        np.testing.assert_array_equal(np.asarray(rf).reshape(few, -1), r[:few])
        np.testing.assert_array_equal(np.asarray(af).reshape(few, -1), a[:few])
