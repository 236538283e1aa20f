"""Worlds where every block of a phase is active, so a wave's block queue is as
full as it gets and all of it lies at one end: sinking blocks only, blocks of
the general form only (the waves of a workgroup share those), and sand that
moves from the first kind to the second."""
import numpy as np
import pytest

import falling_sand_engine_amd as fsg

pytestmark = pytest.mark.gpu

AIR, STONE, SAND, WATER, OIL, STEAM, LAVA, WOOD = range(8)


def dense(kind, W, H, seed):
    rng = np.random.default_rng(seed)
    if kind == "rows":  # sand over air in every block of either row parity
        m = np.where((np.arange(H)[:, None] // 2) % 2 == 0, SAND, AIR) * np.ones((1, W), int)
    else:
        m = rng.choice(kind, size=(H, W))
    c = m.astype(np.uint64) | (np.uint64(320) << np.uint64(16))
    c |= rng.integers(0, 2**32, (H, W), dtype=np.uint64) << np.uint64(32)
    moved = rng.random((H, W)) < 0.5  # sand under way, liquids heading right
    return np.where(moved & np.isin(m, (SAND, WATER, OIL, LAVA)), c | np.uint64(fsg.MOVED), c)


@pytest.mark.parametrize("kind", ["rows", (AIR, SAND), (AIR, WATER), (AIR, STEAM), (OIL, WATER, LAVA), (SAND, STONE),
                                  (AIR, SAND, WATER, STEAM, LAVA, WOOD)])
@pytest.mark.parametrize("W,H", [(64, 64), (2100, 130), (1152, 1024), (2100, 1100)])  # each kernel by world size
@pytest.mark.parametrize("skip", [0, 1])
def test_dense_phases(ctx, orc, kind, W, H, skip):
    print(f"dense {kind} {W}x{H} skip={skip}", flush=True)
    cells = dense(kind, W, H, 7)
    with fsg.World(ctx, W, H, 11, orc.default_config(chunk_skip=skip)) as w:
        w.upload(cells)
        w.tick(5)
        got = w.download()
    ref = orc.run(cells.copy(), orc.default_config(chunk_skip=skip), 11, 0, 5)
    assert np.array_equal(got, ref), int(np.count_nonzero(got != ref))
