"""The reprojection of a given image (no iterations) against the exact transforms
at widths that are no power of two, with both windows: the image's values at the
omitted tilt's nodes, then the adjoint of the projection rows' transform, both as
sums over the nodes in FP64.

Tolerance: the 16-tap interpolation is 1.8e-7 rms of the spectrum's scale, which
for a random image is the line's, three single-precision FFT passes are ~1.5e-7
together and the 1D window 1e-9: 2.4e-7, doubled for the smallest lines.
"""
import numpy as np
import pytest

from feilab_amd import phantom

pytestmark = pytest.mark.gpu


def _exact(img, N, D, plan_nodes):
    X, Y = np.arange(N) - N // 2, np.arange(D) - D // 2
    vx, vy = plan_nodes[:, 0].astype(np.float64), plan_nodes[:, 1].astype(np.float64)
    ex = np.exp(-2j * np.pi * np.outer(vx, X))
    ey = np.exp(-2j * np.pi * np.outer(vy, Y))
    f = np.sum((ex @ img.astype(np.float64)) * ey, 1)
    x = ((np.arange(N) - N / 2.0) / N).astype(np.float32).astype(np.float64)
    return (np.exp(2j * np.pi * np.outer(X, x)) @ f).real


@pytest.mark.parametrize("N,D", [(33, 33), (70, 42), (97, 97), (130, 64), (185, 200), (300, 100), (487, 194), (815, 50)])
@pytest.mark.parametrize("window", ["gauss", "kb6"])
def test_reprojection_of_an_image(icon, oracle_mod, N, D, window):
    tilt = phantom.tilt_series(60, 5)
    plan = icon.Plan(N, tilt, thickness=D, max_slices=2, window=window)
    nodes = oracle_mod.Plan(N, D, tilt, 64).tables()["nodes"].reshape(-1, 2)
    line = nodes[plan.iomit * N:(plan.iomit + 1) * N]
    img = np.random.default_rng(N + D).standard_normal((2, N, D)).astype(np.float32)
    _, rp = plan.solve(np.ones((2, len(tilt), N), np.float32), 0, 0, 0, m_init=img, reproject=True)
    for s in range(2):
        want = _exact(img[s], N, D, line)
        err = np.linalg.norm(rp[s] - want) / np.linalg.norm(want)
        print("reprojection %d x %d, %s: %.1e" % (N, D, window, err), flush=True)
        assert err < 5e-7
