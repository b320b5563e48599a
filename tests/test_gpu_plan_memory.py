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


@pytest.mark.parametrize("N,D,window", [(512, 512, "gauss"), (464, 464, "gauss"), (200, 200, "gauss"), (512, 1000, "gauss"),
                                        (512, 512, "kb6"), (64, 64, "gauss")])
def test_many_slices(icon, N, D, window):
    """A plan for 128 slices and more: the grid rows once, A^H W b, the gradient
    and the reference iterate's (complex, or real at a width that is a power of
    two) and that iterate, and per node the data, the reference's and up to 4
    partials (the weighted values are in the same place)."""
    got, info = _per_slice(icon, N, D, window, 130, 260)
    img, pow2 = N * D, N & (N - 1) == 0
    most = 8 * N * info.n1 + (16 if pow2 else 24) * img + info.M * (16 + 4 * 8) + 32 * N + 16 * info.n1 + 1024
    print("%d x %d, %s: %.3f MB per slice, at most %.3f" % (N, D, window, got / 1e6, most / 1e6), flush=True)
    assert got <= most


@pytest.mark.parametrize("N,D,window", [(64, 64, "gauss"), (100, 40, "gauss"), (128, 64, "kb6"), (90, 200, "gauss")])
def test_fp64_passes_keep_the_bits(icon, N, D, window):
    """131 slices, whose FP64 passes take 66 and 65 of them, against plans that
    take each part at once, and packed with a series of the widest grid."""
    S, it = 131, (2, 9, 3)
    print("two FP64 passes, %d x %d, %s" % (N, D, window), flush=True)
    sino = np.random.default_rng(N).standard_normal((S, len(TILT), N)).astype(np.float32)
    plan = icon.Plan(N, TILT, thickness=D, max_slices=S, window=window)
    m, r, a = plan.solve(sino, *it, 2, 0.0, trace=True)
    part = icon.Plan(N, TILT, thickness=D, max_slices=100, window=window)
    for s in (slice(0, 66), slice(66, S)):
        mp, rp, ap = part.solve(sino[s], *it, 2, 0.0, trace=True)
        np.testing.assert_array_equal(m[s], mp)
        np.testing.assert_array_equal(r[s], rp)
        np.testing.assert_array_equal(a[s], ap)
    wide = icon.Plan(600, TILT, thickness=40, max_slices=1)
    batch = icon.Batch([wide, part, plan], [1, 20, S])
    big = np.random.default_rng(3).standard_normal((1, len(TILT), 600)).astype(np.float32)
    mb, rb, _ = batch.solve([big, sino[:20], sino], *it, trace=True)
    batch.close()
    mw, rw, _ = wide.solve(big, *it, 2, 0.0, trace=True)
    for got, want in zip(mb + rb, (mw, m[:20], m, rw, r[:20], r)):
        np.testing.assert_array_equal(got, np.asarray(want).reshape(got.shape))
