"""Device memory that a plan takes per slice (icon_plan_info.device_bytes of two
capacities), against the sum of the buffers that its kernels use.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

TILT = np.arange(-60, 60.1, 3).astype(np.float32)


def _per_slice(icon, N, D, window, lo, hi):
    out = []
    for S in (lo, hi):
        plan = icon.Plan(N, TILT, thickness=D, max_slices=S, window=window)
        out.append(plan.info.device_bytes)
        info = plan.info
        plan.close()
    return (out[1] - out[0]) / (hi - lo), info


@pytest.mark.parametrize("N,D,window", [(1007, 1007, "gauss"), (1024, 600, "gauss"), (700, 300, "kb6")])
def test_widest_grid(icon, N, D, window):
    """n0 = 2048, where no gradient is computed in FP64: grid rows, A^H W b and
    gradient, and per node the data, up to 4 partials and 3 weighted values."""
    got, info = _per_slice(icon, N, D, window, 4, 8)
    assert info.n0 == 2048
    img = N * D
    most = 8 * N * info.n1 + 12 * img + info.M * (8 + 4 * 8 + 3 * 8) + 16 * N + 16 * info.n1 + 1024
    print("%d x %d, %s: %.2f MB per slice, at most %.2f" % (N, D, window, got / 1e6, most / 1e6), flush=True)
    assert got <= most
