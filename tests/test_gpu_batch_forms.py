"""Batches whose worlds share a setting run a tick kernel compiled for it (the
skipping ones over one list of the awake chunks of all worlds); batches whose
worlds differ, or have a tick zone, the one that reads each world's setting.
Every form equals stepping each world alone."""
import numpy as np
import pytest

import falling_sand_engine_amd as fsg

pytestmark = pytest.mark.gpu

SIZES = [(64, 64), (65, 130), (200, 63), (448, 320), (1000, 130)]
LARGE = SIZES + [(2500, 2100)]  # more chunks than can be resident at once: the awake ones are listed


def batch_of(ctx, skips, reacts, zoned, sizes=SIZES):
    worlds = []
    for i, (W, H) in enumerate(sizes):
        cfg = fsg.default_config(chunk_skip=skips[i % len(skips)], reactions=reacts[i % len(reacts)])
        w = fsg.World(ctx, W, H, 40 + i, cfg)
        w.generate(4, 40 + i)
        if zoned and i == 2:
            w.tickZone = (7, 9, W - 20, H - 12)
        worlds.append(w)
    return worlds


@pytest.mark.parametrize("skips,reacts,zoned", [
    ((0,), (0,), False), ((0,), (1,), False), ((1,), (0,), False), ((1,), (1,), False),  # one setting each
    ((0, 1), (1,), False), ((1,), (0, 1), False), ((1,), (1,), True), ((0,), (0,), True)])  # the general form
@pytest.mark.parametrize("sizes", [SIZES, LARGE])
@pytest.mark.parametrize("ticks", [(16, 5, 32), (1, 3)])
def test_batch_form_equals_alone(ctx, skips, reacts, zoned, sizes, ticks):
    print(f"batch form skips={skips} reacts={reacts} zoned={zoned} worlds={len(sizes)} ticks={ticks}", flush=True)
    together, alone = batch_of(ctx, skips, reacts, zoned, sizes), batch_of(ctx, skips, reacts, zoned, sizes)
    for n in ticks:  # graphs, an odd remainder (the list's counts go by tick parity), and graphs again
        fsg.batch_step(ctx, together, n)
        for w in alone:
            w.tick(n)
    for a, b in zip(together, alone):
        assert np.array_equal(a.download(), b.download()), (a.width, a.height)
        a.close()
        b.close()


def test_batch_form_changes_between_calls(ctx):
    """A cached graph is not replayed for another form: the zone set between
    two calls takes the same worlds from the listed to the general form."""
    together, alone = batch_of(ctx, (1,), (1,), False, LARGE), batch_of(ctx, (1,), (1,), False, LARGE)
    for zone in (None, (3, 5, 300, 200), (0, 0, 448, 320)):
        if zone:
            together[3].tickZone = alone[3].tickZone = zone
        fsg.batch_step(ctx, together, 32)
        for w in alone:
            w.tick(32)
        for a, b in zip(together, alone):
            assert np.array_equal(a.download(), b.download()), (zone, a.width)
    for w in together + alone:
        w.close()


@pytest.mark.parametrize("first,second", [(SIZES[:2], SIZES[2:]), (SIZES, SIZES[:1])])  # more worlds then, and fewer
@pytest.mark.parametrize("skip", [0, 1])
def test_a_batch_too_short_for_a_graph_leaves_the_cached_one_alone(ctx, first, second, skip):
    """A graph captured over one set of worlds is not replayed for another set
    whose last call had fewer ticks than a graph has."""
    print(f"graph of {len(first)} worlds, then {len(second)} others, skip={skip}", flush=True)
    a, b, alone = (batch_of(ctx, (skip,), (1,), False, s) for s in (first, second, second))
    fsg.batch_step(ctx, a, 16)
    for n in (5, 16, 33):
        fsg.batch_step(ctx, b, n)
        for w in alone:
            w.tick(n)
        for x, y in zip(b, alone):
            assert np.array_equal(x.download(), y.download()), (n, x.width, x.height)
    ref = [w.download() for w in a]
    for w in b:
        w.close()
    fsg.batch_step(ctx, a, 16)  # the first set's own graph or a new one
    again = batch_of(ctx, (skip,), (1,), False, first)
    fsg.batch_step(ctx, again, 32)
    for x, y, r in zip(a, again, ref):
        assert not np.array_equal(r, x.download()) and np.array_equal(x.download(), y.download())
    for w in a + alone + again:
        w.close()
