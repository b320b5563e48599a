"""icon_preprocess over stack shapes, against the oracle: one image and many,
images smaller than a block and of several blocks with a ragged last round,
constant images, an image whose extreme pixel lies outside the central region.

The modes and the mode-subtracted images are bit-identical (the same double
arithmetic, an integer histogram); the normalised images differ by the order
of the FP64 sums and one rounding of the factor: 2 ulp of single precision,
and 2e-6 of the largest value allows for the reference's own mean, summed from
single-precision quotients.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SHAPES = [(1, 1, 1), (1, 3, 7), (3, 16, 16), (2, 45, 46), (1, 300, 257), (40, 33, 65), (7, 128, 513), (1, 700, 1000)]


@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "%dx%dx%d" % s)
def test_preprocess_shapes(icon, oracle_mod, shape):
    nz, ny, nx = shape
    print("preprocess %d images of %d x %d" % (nz, ny, nx), flush=True)
    rng = np.random.default_rng(nz + ny * nx)
    st = (rng.gamma(4.0, 30.0, shape) + 20 * rng.standard_normal((nz, 1, 1))).astype(np.float32)
    st[0, 0, 0] = 5e4   # outside the central region where there is a border
    out, modes = icon.icon.preprocess(st)
    ref, rmodes = oracle_mod.preprocess(st)
    np.testing.assert_array_equal(modes, rmodes)
    np.testing.assert_array_equal(out, ref)
    if ny * nx > 1:
        tilt = np.linspace(-60, 60, nz).astype(np.float32)
        out, modes = icon.icon.preprocess(st, tilt, 200)
        ref, rmodes = oracle_mod.preprocess(st, tilt, 200)
        np.testing.assert_array_equal(modes, rmodes)
        np.testing.assert_allclose(out, ref, rtol=2e-6, atol=2e-6 * np.abs(ref).max())


def test_preprocess_constant_images(icon, oracle_mod):
    print("preprocess constant images", flush=True)
    st = np.full((2, 50, 60), 7.25, np.float32)
    out, modes = icon.icon.preprocess(st)
    np.testing.assert_array_equal(modes, [7.25, 7.25])
    np.testing.assert_array_equal(out, np.zeros_like(st))
