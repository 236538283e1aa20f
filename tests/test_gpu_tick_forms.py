"""The tick of worlds without skipping that take more than one chunk per
compute unit, on either side of the lines between its forms, against the
oracle.  The sizes follow from the number of compute units, 256."""
import numpy as np
import pytest

import falling_sand_engine_amd as fsg

pytestmark = pytest.mark.gpu


def random_mix(W, H, seed):
    """Every material, hot cells (burning wood, reactions), MOVED flags."""
    rng = np.random.default_rng(seed)
    mats = rng.choice(8, size=(H, W), p=[.35, .1, .2, .12, .08, .07, .05, .03]).astype(np.uint64)
    cells = mats | (rng.integers(0, 700 * 16, size=(H, W)).astype(np.uint64) << np.uint64(16))
    cells |= rng.integers(0, 2**32, size=(H, W), dtype=np.uint64) << np.uint64(32)
    return cells | ((rng.integers(0, 2, size=(H, W)) * (mats == 2)).astype(np.uint64) << np.uint64(8))


def check(ctx, orc, W, H, cfg, ticks, zone=None, seed=31):
    print(f"tick form {W}x{H} cell_iter={cfg.cell_iter} reactions={cfg.reactions} zone={zone}", flush=True)
    cells = random_mix(W, H, seed)
    with fsg.World(ctx, W, H, seed, cfg) as w:
        w.upload(cells)
        if zone:
            w.tickZone = zone
        w.tick(ticks)
        got = w.download()
    ref = orc.run(cells, cfg, seed, 0, ticks, zone)
    assert np.array_equal(got, ref), np.argwhere(got != ref)[:3]


@pytest.mark.parametrize("W,H", [(4096, 4096), (4160, 4096)])  # the last is past the last-level cache
def test_one_phase_of_large_worlds(ctx, orc, W, H):
    """One phase a tick: six workgroups per CU (1,536 at once, 1,024 chunks
    left over) and five (1,280 at once, 320 left over, which run as quarters)."""
    check(ctx, orc, W, H, orc.default_config(cell_iter=1), 3)
