"""Outlines where the batched walks can go wrong: many small loops that meet
(saddles, shared corners, the clamped last row and column), loops of around
64 runs, which a lane's walk has no room for, loops of thousands of runs, and
regions too long for the lanes' walks."""
import numpy as np
import pytest

import falling_sand_engine_amd as fsg

pytestmark = pytest.mark.gpu

SHAPES = [(128, 128), (255, 64), (64, 255), (127, 129), (300, 50), (16384, 1), (2000, 8), (9, 1800), (33, 65), (2, 2)]


def solid(kind, w, h, seed):
    rng = np.random.default_rng(seed)
    y, x = np.mgrid[0:h, 0:w]
    if kind == "comb":  # teeth of a comb: one loop of four runs per tooth
        return (x % 2 == 0) | (y == h // 2)
    if kind == "combs":  # separate combs of 15 and 16 teeth: 62 to 66 runs each
        return ((x % 33 % 2 == 0) & (x % 33 < 31) & (y % 7 < 4)) | ((y % 7 == 3) & (x % 33 < 31))
    if kind == "checker":
        return (x + y) % 2 == 0
    if kind == "full":
        return np.ones((h, w), bool)
    if kind == "rings":
        return np.maximum(abs(x - w // 2), abs(y - h // 2)) % 4 < 2
    return rng.random((h, w)) < kind


@pytest.mark.parametrize("kind", [0.03, 0.2, 0.5, 0.6, 0.9, "comb", "combs", "checker", "full", "rings"])
def test_mesh_batches_match_oracle(ctx, orc, kind):
    cfg = orc.default_config()
    for k, (w, h) in enumerate(SHAPES):
        print(f"mesh batch {kind} {w}x{h}", flush=True)
        m = solid(kind, w, h, 10 * k)
        W, H = min(w + 6, 16384), h + 5  # the region ends before the world's last row and column
        if w + 6 > W:
            m = m[:, :W - 3]
        rw, rh = m.shape[1], m.shape[0]
        cells = np.full((H, W), fsg.make_cell(fsg.MAT_AIR, 320), dtype=np.uint64)
        cells[2:2 + rh, 1:1 + rw][m] = fsg.make_cell(fsg.MAT_STONE, 320, 0xFF808080)
        with fsg.World(ctx, W, H, 1, cfg) as world:
            world.upload(cells)
            got = world.mesh([(1, 2, rw, rh)])
        assert got[0][0] == 0
        want = orc.mesh_mask(m.astype(np.uint8))
        assert got[0][1] == want, (kind, w, h, len(got[0][1]), len(want))
