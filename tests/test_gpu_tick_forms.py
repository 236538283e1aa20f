"""The tick of worlds without skipping that take more than one chunk per
compute unit, on either side of the lines between its forms, against the
oracle.  The sizes follow from the number of compute units, 256, and each test
says which chunks it means to run in which form."""
import ctypes

import numpy as np
import pytest

import falling_sand_engine_amd as fsg

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def cu():
    """Compute units of the device (hipDeviceAttributeMultiprocessorCount)."""
    n = ctypes.c_int()
    assert ctypes.CDLL("libamdhip64.so.7").hipDeviceGetAttribute(ctypes.byref(n), 63, 0) == 0
    return n.value


def chunks(W, H):
    return -(-W // 64) * -(-H // 64)


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


# 40 x 39 = 1,560 chunks, 24 past the 1,536 resident at once: those run as quarters
@pytest.mark.parametrize("cell_iter", [1, 2, 3])
@pytest.mark.parametrize("react", [0, 1])
@pytest.mark.parametrize("trim", [0, 13])  # the last chunks whole and ragged
def test_chunks_past_a_round_run_as_quarters(ctx, orc, cu, cell_iter, react, trim):
    W, H = 2560 - trim, 2496 - trim
    assert 0 < chunks(W, H) % (6 * cu) <= 6 * cu // 4 and chunks(W, H) > 6 * cu
    check(ctx, orc, W, H, orc.default_config(cell_iter=cell_iter, reactions=react), 5)


# 36 x 36 = 1,296 chunks, 16 past the 1,280 resident at once with zone tests,
# all in the last row of chunks: the zone ends before it, inside it and past it
@pytest.mark.parametrize("cell_iter", [1, 3])
@pytest.mark.parametrize("zone", [(100, 3, 2100, 2200), (70, 64, 2101, 2207), (1290, 90, 801, 2200), (0, 1, 2304, 2303)])
def test_quarters_with_a_zone(ctx, orc, cu, cell_iter, zone):
    W = H = 2304
    assert 0 < chunks(W, H) % (5 * cu) <= 5 * cu // 4 and chunks(W, H) > 5 * cu
    check(ctx, orc, W, H, orc.default_config(cell_iter=cell_iter), 5, zone)


def test_quarters_with_nine_materials(ctx, orc, cu):
    """More materials than the class tables hold: pair tables throughout."""
    W, H, seed = 2560, 2496, 5
    cfg = orc.default_config()
    cfg.n_materials = 9
    cfg.materials[8] = cfg.materials[fsg.MAT_SAND]
    cells = random_mix(W, H, seed)
    cells[::3] |= np.uint64(8) * ((cells[::3] & np.uint64(15)) == 0)
    print("tick form nine materials", flush=True)
    with fsg.World(ctx, W, H, seed, cfg) as w:
        w.upload(cells)
        w.tick(4)
        got = w.download()
    assert np.array_equal(got, orc.run(cells, cfg, seed, 0, 4))


# 20 x 20 = 400 chunks of 512 threads, 24 x 24 = 576 of 256
@pytest.mark.parametrize("W,H", [(1280, 1280), (1270, 1219), (1536, 1536)])
@pytest.mark.parametrize("react", [0, 1])
@pytest.mark.parametrize("zone", [None, (67, 5, 1100, 1190), (640, 640, 1, 1)])
def test_worlds_of_a_few_chunks_per_compute_unit(ctx, orc, cu, W, H, react, zone):
    assert (cu < chunks(W, H) <= 2 * cu) == (W < 1500) and chunks(W, H) <= 5 * cu
    check(ctx, orc, W, H, orc.default_config(reactions=react), 6, zone)


@pytest.mark.parametrize("W,H", [(4096, 4096), (4160, 4096)])  # the last is past the last-level cache
def test_one_phase_of_large_worlds(ctx, orc, W, H):
    """One phase a tick: six workgroups per CU (1,536 at once, 1,024 chunks
    left over) and five (1,280 at once, 320 left over, which run as quarters)."""
    check(ctx, orc, W, H, orc.default_config(cell_iter=1), 3)
