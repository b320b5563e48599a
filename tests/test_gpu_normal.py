"""The solve's normal operator (its kernel's spectrum on the oversampled grid,
the 16-tap interpolation of the residual's node values, the gradient energy)
against the FP64 oracle's NUFFT iteration, at the edges of its grids and
tiles: the smallest width, a width that fills the grid, odd widths, thickness
and width on different grids, tilts up to +-90 degrees, few tilts.

Tolerances: the oracle iterates a 14-tap Gaussian NUFFT whose error is 7e-7
rms and 3.5e-6 at most of the transform's scale; single-precision FFTs add
~3e-7.  Eight descent steps at most multiply a relative error by the number
of steps, so 3e-5 bounds the image, and 1e-5 the residual norm (an error of
the iterate enters the residual at second order) and the step sizes' ratio of
two quadratic forms.
"""
import numpy as np
import pytest

from feilab_amd import phantom

pytestmark = pytest.mark.gpu

CASES = [
    # N, thickness, tilts
    (33, 33, np.linspace(-60, 60, 9)),
    (64, 64, np.linspace(-60, 60, 21)),
    (64, 40, np.linspace(-90, 90, 13)),
    (65, 200, np.linspace(-57, 63, 11)),
    (128, 128, np.linspace(-70, 70, 5)),
    (129, 90, np.linspace(-45, 60, 15)),
    (256, 64, np.linspace(-60, 60, 7)),
    (300, 517, np.linspace(-60, 60, 6)),
]


def _sino(N, nz, seed):
    rng = np.random.default_rng(seed)
    x = rng.standard_normal((2, nz, N)).astype(np.float32)
    return (x + 2 * np.exp(-((np.arange(N) - N / 2) / 9.0) ** 2)).astype(np.float32)


@pytest.mark.parametrize("case", CASES, ids=lambda c: "%dx%d_%d" % (c[0], c[1], len(c[2])))
def test_normal_operator_solve_vs_fp64_oracle(icon, oracle_mod, case):
    N, D, tilt = case
    tilt = np.asarray(tilt, np.float32)
    print("normal operator %dx%d, %d tilts" % (N, D, len(tilt)), flush=True)
    sino = _sino(N, len(tilt), N + D)
    plan = icon.Plan(N, tilt, thickness=D, max_slices=2)
    m, rp, res, al = plan.solve(sino, 2, 4, 2, 2, 0.0, trace=True, reproject=True)
    orc = oracle_mod.Plan(N, D, tilt, 64)
    for s in range(2):
        mo, reso, alo = orc.solve(sino[s], 2, 4, 2, 2, 0.0, trace=True)
        err = np.linalg.norm(m[s] - mo) / np.linalg.norm(mo)
        print("  slice %d: image %.1e, residual %.1e, alpha %.1e" %
              (s, err, np.abs(res[s] / reso - 1).max(), np.abs(al[s] / alo - 1).max()), flush=True)
        assert err < 3e-5
        assert np.abs(res[s] / reso - 1).max() < 1e-5
        assert np.abs(al[s] / alo - 1).max() < 1e-5
        ro = orc.reproject(mo)
        assert np.linalg.norm(rp[s] - ro) / np.linalg.norm(ro) < 3e-5


@pytest.mark.parametrize("N", [64, 97])
def test_solve_is_the_same_without_residuals_and_as_a_graph(icon, N):
    print("solve with and without residuals, width %d" % N, flush=True)
    tilt = phantom.tilt_series(60, 6)
    sino = _sino(N, len(tilt), N)
    plan = icon.Plan(N, tilt, max_slices=2)
    m, res, al = plan.solve(sino, 1, 3, 1, 2, 0.0, trace=True)
    np.testing.assert_array_equal(plan.solve(sino, 1, 3, 1, 2, 0.0), m)
    for _ in range(3):
        mg, rg, ag = plan.solve(sino, 1, 3, 1, 2, 0.0, trace=True, use_graph=True)
        np.testing.assert_array_equal(mg, m)
        np.testing.assert_array_equal(rg, res)
        np.testing.assert_array_equal(ag, al)
    one = plan.solve(sino[:1], 1, 3, 1, 2, 0.0)
    np.testing.assert_array_equal(one, m[:1])
