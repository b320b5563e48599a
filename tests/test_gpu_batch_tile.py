"""A packed solve's captured graph outlives changes of its plans' column tile:
the tile is set to another width and back, with other allocations in between
that take freed memory, and to the width that it has; the next solves, with
the plans' tables at either width, must give the first one's bits.  The batch
autotuner tunes every plan's transforms, 6-tap ones too, and leaves the packed
solve's bits.
"""
import numpy as np
import pytest

from feilab_amd import phantom

pytestmark = pytest.mark.gpu


def test_packed_solve_after_tile_changes(icon):
    from feilab_amd.icon import DeviceArray, SolveOptions
    print("packed solve before and after set_col_block", flush=True)
    cfg = [(200, "gauss"), (512, "gauss"), (256, "kb6"), (300, "kb6")]
    tilt, rng, S, it = phantom.tilt_series(60, 4), np.random.default_rng(77), 2, (1, 3, 1)
    plans = [icon.Plan(N, tilt, max_slices=S, window=w) for N, w in cfg]
    batch = icon.Batch(plans, [S] * len(plans))
    d_s = [DeviceArray.from_host(rng.standard_normal((S, len(tilt), N)).astype(np.float32)) for N, _ in cfg]
    d_m = [DeviceArray((S, N, N), np.float32) for N, _ in cfg]
    d_r = [DeviceArray((S, sum(it) + 1), np.float64) for _ in cfg]
    opts = SolveOptions(*it, 2, 0.0, 1, 0)

    def solve():
        batch.reconstruct_dev(d_s, d_m, opts, d_resids=d_r)
        icon.lib().icon_device_synchronize()
        return [d.numpy() for d in d_m] + [d.numpy() for d in d_r]

    first = solve()
    held = []
    for tiles in ((16, 16, 8, 8), (8, 8, 8, 8), (16, 8, 8, 8)):
        for p, t in zip(plans, tiles):
            p.set_col_block(t)
            held += [DeviceArray.from_host(np.full(n, np.nan, np.float32)) for n in (1 << 10, 1 << 14, 1 << 18, 1 << 20)]
        for a, b in zip(solve(), first):
            np.testing.assert_array_equal(a, b)
        print("  tiles %s: same bits" % (tiles,), flush=True)
    with pytest.raises(icon.IconError):
        plans[2].set_col_block(16)
    batch.close()


def test_batch_autotune_keeps_bits(icon):
    print("packed solve before and after the batch autotuner", flush=True)
    cfg = [(200, "gauss"), (512, "gauss"), (900, "gauss"), (256, "kb6"), (256, "gauss")]
    tilt, rng, S = phantom.tilt_series(60, 4), np.random.default_rng(78), 2
    plans = [icon.Plan(N, tilt, max_slices=S, window=w) for N, w in cfg]
    sinos = [rng.standard_normal((S, len(tilt), N)).astype(np.float32) for N, _ in cfg]
    batch = icon.Batch(plans, [S] * len(plans))
    before = batch.solve(sinos, 2, 4, 2, trace=True)
    tiles = batch.autotune()
    print("  tiles", tiles, flush=True)
    assert all(t in ((8, 16) if N <= 512 and w == "gauss" else (8,)) for t, (N, w) in zip(tiles, cfg))
    assert [p.info.col_block for p in plans] == tiles
    after = batch.solve(sinos, 2, 4, 2, trace=True)
    for k in (0, 1):
        for a, b in zip(after[k], before[k]):
            np.testing.assert_array_equal(a, b)
    batch.close()
