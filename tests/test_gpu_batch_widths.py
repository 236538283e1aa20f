"""Batches of few chunks take wider workgroups: on either side of the lines
between 1024, 512 and 256 threads per chunk each world equals the one ticked
alone, with skipping and without."""
import numpy as np
import pytest

import falling_sand_engine_amd as fsg

from test_gpu_batch_forms import batch_of

pytestmark = pytest.mark.gpu

# chunks: 1, 256 | 257, 512 | 513, 896 | 897
SIZES = [[(33, 20)], [(1000, 1000)], [(64, 64), (1024, 1024)], [(2048, 1000)], [(1024, 2048), (7, 64)],
         [(1024, 1024), (2560, 1024)], [(3580, 1020), (64, 1)]]


@pytest.mark.parametrize("sizes", SIZES)
@pytest.mark.parametrize("skip,react", [(0, 0), (0, 1), (1, 0), (1, 1)])
def test_batch_width_equals_alone(ctx, sizes, skip, react):
    print(f"batch width {sizes} skip={skip} react={react}", flush=True)
    together, alone = batch_of(ctx, (skip,), (react,), False, sizes), batch_of(ctx, (skip,), (react,), False, sizes)
    for n in (17, 3):
        fsg.batch_step(ctx, together, n)
        for w in alone:
            w.tick(n)
    for a, b in zip(together, alone):
        assert np.array_equal(a.download(), b.download()), (a.width, a.height)
        assert a.stats().tiles_processed == b.stats().tiles_processed
        a.close()
        b.close()


# a batch below the lines, one above the line without skipping only, one above both
@pytest.mark.parametrize("sizes,wide", [([(320, 256)] * 3, (0, 1)), ([(2048, 1280)], (1,)), ([(4096, 2048)], ())])
def test_autotune_where_the_register_budget_does_not_apply(ctx, sizes, wide):
    """The budget is the 256-thread kernel's: candidates that differ only in it
    have one time where the batch takes wider workgroups (`wide`: the skip
    settings with which it does), and the choice is then the default."""
    worlds = batch_of(ctx, (1,), (1,), False, sizes)
    print(f"autotune {sizes}", flush=True)
    rep = ctx.autotune(worlds, sample_ticks=8)
    ctx.set_tuning()
    for w in worlds:
        w.close()
    assert not rep["from_cache"]
    ms = {(c["graph_ticks"], c["chunk_skip"], c["occupancy"]): c["ms"] for c in rep["candidates"]}
    assert len(ms) == 20 and min(ms.values()) > 0
    for skip in (0, 1):
        same = [ms[t, skip, 4] == ms[t, skip, 5] for t in (1, 4, 8, 16, 32)]
        assert all(same) if skip in wide else not all(same), (skip, same)
    assert rep["best"]["chunk_skip"] not in wide or rep["best"]["occupancy"] == 5
