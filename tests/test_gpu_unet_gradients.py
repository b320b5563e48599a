"""Parameter gradients of the warm-start U-Net at sizes on the edges of the
backward kernels' tiles: one pixel per image at the deepest level, widths that
are no multiple of the 16-pixel strips, heights that end inside a row segment,
several images per split.  Tolerance: as test_unet_gradients_vs_oracle, twice
what BF16 rounding alone moves a block, at least 1e-2.
"""
import numpy as np
import pytest

from test_gpu_unet import _blocks, _net_and_params, rel

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", [(1, 8, 8), (3, 24, 40), (2, 136, 72), (1, 40, 152), (5, 64, 16)])
def test_gradients_at_tile_edges(icon, shape):
    from oracle import unet_ref
    B, H, W = shape
    print("unet gradients", shape, flush=True)
    net, p = _net_and_params(H, W, B + 1, seed=H + W)
    rng = np.random.default_rng(H * W + B)
    x = rng.standard_normal(shape).astype(np.float32)
    t = (0.5 * x + 0.1 * rng.standard_normal(shape)).astype(np.float32)
    loss, g = net.gradients(x, t)
    rloss, rg = unet_ref.gradients(p, x, t, bf16=True)
    _, rg64 = unet_ref.gradients(p, x, t, bf16=False)
    assert abs(loss - rloss) <= 1e-2 * abs(rloss)
    for name, a, b in _blocks():
        gd, gr, g64 = g[a:b].astype(np.float64), rg[a:b], rg64[a:b]
        if np.linalg.norm(gr) == 0:
            assert np.linalg.norm(gd) == 0, name
            continue
        assert rel(gd, gr) <= max(2.0 * rel(gr, g64), 1e-2), (name, rel(gd, gr), rel(gr, g64))
    # the same call again: every sum is taken in a fixed order
    _, g2 = net.gradients(x, t)
    np.testing.assert_array_equal(g, g2)
    net.close()
