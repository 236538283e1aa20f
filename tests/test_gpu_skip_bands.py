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
