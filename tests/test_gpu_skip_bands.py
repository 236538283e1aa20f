"""Chunk skipping with the wake test in each workgroup, of 1024, 512 and 256
threads, and over the list: on either side of the lines between the forms
each equals the oracle (which has no skipping), with whole and ragged last
chunks, a tick zone, and cells set while chunks sleep."""
import numpy as np
import pytest

import falling_sand_engine_amd as fsg

pytestmark = pytest.mark.gpu

# chunks across and down: 1, 256 | 258 .. 896 | 897 .. 2560 | 2561 chunks
BANDS = [(1, 1), (16, 16), (43, 6), (64, 14), (299, 3), (64, 40), (197, 13)]


def mostly_asleep(tx, ty, trim):
    """A world of air and stone with a pile of sand and water here and there."""
    W, H = tx * 64 - trim, ty * 64 - (trim and 5)
    rng = np.random.default_rng(tx * 100 + ty)
    cells = np.full((H, W), fsg.make_cell(fsg.MAT_AIR, 320, 0), np.uint64)
    cells[-3:] = fsg.make_cell(fsg.MAT_STONE, 320, 1)
    for _ in range(max(2, tx * ty // 12)):
        x, y = int(rng.integers(0, W)), int(rng.integers(0, H))
        cells[y:y + 20, x:x + 9] = fsg.make_cell(int(rng.choice([fsg.MAT_SAND, fsg.MAT_WATER])),
                                                 int(rng.integers(300, 340)), int(rng.integers(0, 2**32)))
    return cells


@pytest.mark.parametrize("tx,ty", BANDS)
@pytest.mark.parametrize("react,trim,zoned", [(1, 0, 0), (0, 0, 0), (1, 11, 0), (1, 0, 1)])
def test_skip_forms_equal_oracle(ctx, orc, tx, ty, react, trim, zoned):
    print(f"skip form {tx}x{ty} react={react} trim={trim} zoned={zoned}", flush=True)
    cells = mostly_asleep(tx, ty, trim)
    H, W = cells.shape
    cfg = orc.default_config(chunk_skip=1, reactions=react)
    zone = (W // 5, 3, W // 2 + 1, H - 10) if zoned else None
    with fsg.World(ctx, W, H, 9, cfg) as w:
        w.upload(cells)
        if zone:
            w.tickZone = zone
        ref = cells
        for t, n in ((0, 3), (3, 4)):
            w.tick(n)
            ref = orc.run(ref.copy(), cfg, 9, t, n, zone)
            assert np.array_equal(w.download(), ref), t
            x, y = W // 2, H // 3  # a cell set in a chunk that may sleep
            w.setTile(x, y, fsg.make_cell(fsg.MAT_SAND, 320, 5))
            ref[y, x] = fsg.make_cell(fsg.MAT_SAND, 320, 5)
        st = w.stats()
        assert zoned or tx * ty < 200 or st.tiles_processed < st.tiles_offered


@pytest.mark.parametrize("zoned", [0, 1])
def test_listed_world_across_jumps_and_batches(ctx, orc, zoned):
    """2,561 chunks are the fewest whose awake ones are listed by tick parity:
    ticks run by the batch path, or a jump of the tick counter by an odd or
    even number, in between listed ticks."""
    tx, ty = BANDS[-1]
    cells = mostly_asleep(tx, ty, 0)
    H, W = cells.shape
    assert -(-W // 64) * -(-H // 64) == 2561
    cfg = orc.default_config(chunk_skip=1)
    zone = (W // 7, 0, W // 2, H - 70) if zoned else None
    print(f"listed world across jumps zoned={zoned}", flush=True)
    with fsg.World(ctx, W, H, 9, cfg) as w:
        w.upload(cells)
        if zone:
            w.tickZone = zone
        ref, t = cells, 0
        for jump, how, n in ((0, "tick", 3), (0, "batch", 2), (0, "tick", 2), (0, "batch", 3), (0, "tick", 1),
                             (51, "tick", 3), (30, "tick", 2), (0, "batch", 1), (7, "batch", 2), (1, "tick", 3)):
            if jump:
                t += jump
                w.set_tick(t)
            w.tick(n) if how == "tick" else fsg.batch_step(ctx, [w], n)
            ref = orc.run(ref, cfg, 9, t, n, zone)
            t += n
            assert np.array_equal(w.download(), ref), (t, how)
        assert zoned or w.stats().tiles_processed < w.stats().tiles_offered
