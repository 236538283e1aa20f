"""Islands at the edges of the search's window of 64 x 64 cells around the seed
against the oracle: bars that end inside, at and past its sides, shapes that
leave the window and come back, windings, blocks of 1000 cells and one more,
and seeds by the grid's corners."""
import numpy as np
import pytest

import falling_sand_engine_amd as fsg
from test_gpu_islands import compare

pytestmark = pytest.mark.gpu

STONE = fsg.make_cell(fsg.MAT_STONE, 300, 0xFF445566)
AIR = fsg.make_cell(fsg.MAT_AIR, 320, 0)


def check(ctx, orc, c, seeds):
    cfg = orc.default_config()
    with fsg.World(ctx, c.shape[1], c.shape[0], 1, cfg) as w:
        w.upload(c)
        got = w.physicsCheck(seeds)
        grid = w.download()
    ref = c.copy()
    compare(got, orc.physics_check(ref, cfg, seeds))
    assert np.array_equal(grid, ref)


@pytest.mark.parametrize("reach", [30, 31, 32, 33, 40])
@pytest.mark.parametrize("dx,dy", [(1, 0), (-1, 0), (0, 1), (0, -1)])
def test_bars(ctx, orc, reach, dx, dy):
    c = np.full((150, 170), AIR, np.uint64)
    for k in range(reach + 1):
        c[75 + k * dy, 85 + k * dx] = STONE
    check(ctx, orc, c, [(85, 75), (85 + reach * dx, 75 + reach * dy)])


@pytest.mark.parametrize("W,H", [(200, 150), (63, 40), (64, 64), (65, 70)])
def test_windings_hooks_and_corners(ctx, orc, W, H):
    c = np.full((H, W), AIR, np.uint64)
    c[0:H - 2:4, 1:W - 1] = STONE              # a winding over the whole grid, too large
    c[2:H - 2:8, W - 2] = STONE
    c[0, 0] = STONE
    seeds = [(0, 0), (W - 1, H - 1), (W // 2, 0), (W - 2, 4 % H), (1, H - 1)]
    check(ctx, orc, c, seeds)
    c = np.full((H, W), AIR, np.uint64)
    for k, x in enumerate(range(0, min(W, 40), 4)):  # windings of at most 1000 cells
        c[0:min(H, 60), x] = STONE
        if x + 4 < min(W, 40):
            c[0 if k % 2 else min(H, 60) - 1, x:x + 5] = STONE
    c[H - 1, W - 12:] = STONE
    check(ctx, orc, c, [(0, 0), (W - 1, H - 1), (4, 7)])


@pytest.mark.parametrize("n", [9, 10, 11, 999, 1000, 1001])
def test_block_sizes(ctx, orc, n):
    c = np.full((128, 128), AIR, np.uint64)
    idx = np.arange(n)
    c[50 + idx // 40, 40 + idx % 40] = STONE
    check(ctx, orc, c, [(40, 50), (45, 50)])


def test_hook_leaves_the_window_and_comes_back(ctx, orc):
    c = np.full((160, 200), AIR, np.uint64)
    c[60, 60:140] = STONE
    c[60:80, 139] = STONE
    c[79, 60:140] = STONE
    check(ctx, orc, c, [(62, 79), (60, 60)])
    c[79, 100] = AIR  # now two hooks, one from each side
    check(ctx, orc, c, [(99, 79), (101, 79)])


def winding(n, side, spiral):
    """The first n cells of a path one cell wide: rows of `side` cells joined at
    alternating ends, or a spiral inwards."""
    if not spiral:
        path = [(x if (r & 1) == 0 else side - 1 - x, 2 * r + d)
                for r in range(n) for x, d in [(x, 0) for x in range(side)] + [(side - 1, 1)]]
        return path[:n]
    x, y, dx, dy, leg, path = 0, 0, 1, 0, side - 1, []
    turns = 0
    while len(path) < n and leg > 0:
        for _ in range(leg):
            path.append((x, y))
            x, y = x + dx, y + dy
        dx, dy = -dy, dx
        turns += 1
        if turns >= 3 and turns % 2:
            leg -= 2
    return path[:n]


@pytest.mark.parametrize("n", [999, 1000, 1001, 1400])
@pytest.mark.parametrize("side,spiral", [(40, 0), (60, 0), (12, 0), (58, 1)])
@pytest.mark.parametrize("turned", [0, 1])
def test_long_windings(ctx, orc, n, side, spiral, turned):
    """Windings at the size limit and past it, within one window and (12 cells
    wide) longer than it, which take a fill step a row or more."""
    W, H = 260, 250
    c = np.full((H, W), AIR, np.uint64)
    path = winding(n, side, spiral)
    assert len(set(path)) == n
    path = [(y, x) if turned else (x, y) for x, y in path]
    for x, y in path:
        c[10 + y, 15 + x] = STONE
    seeds = [(15 + path[k][0], 10 + path[k][1]) for k in (0, n // 2, n - 1)]
    print(f"winding n={n} side={side} spiral={spiral} turned={turned}", flush=True)
    for s in seeds:
        ref = orc.physics_check(c.copy(), orc.default_config(), [s])[0]
        assert (ref["status"] == fsg._abi.ISLAND_BODY) == (n <= 1000) and (n > 1000 or ref["count"] == n)
        check(ctx, orc, c, [s])


@pytest.mark.parametrize("W,H", [(200, 150), (63, 40), (64, 64), (65, 70)])
def test_winding_over_the_whole_grid(ctx, orc, W, H):
    c = np.full((H, W), AIR, np.uint64)
    rows = range(0, H - 6, 2)
    for k, y in enumerate(rows):
        c[y, 1:W - 1] = STONE
        c[y:y + 3, W - 2 if k % 2 else 1] = STONE
    seeds = [(1, 0), (W // 2, 0), (W - 2, 4), (W // 2, H - 8), (0, H - 1)]
    ref = orc.physics_check(c.copy(), orc.default_config(), seeds)
    assert [r["status"] for r in ref].count(fsg._abi.ISLAND_ATTACHED) == 4
    check(ctx, orc, c, seeds)
