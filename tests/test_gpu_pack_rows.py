"""The encoder's wave-parallel row parse against the oracle's, on records that
reach its edges: rows with no match (literals carried over many of them, to
the next row with one or to the block's end), rows that are one run, runs cut
by the lanes' and rows' ends, short runs that stay literals, and both ways a
byte can repeat at once."""
import numpy as np
import pytest

import falling_sand_engine_amd as fsg
from test_gpu_pack import oracle_images

pytestmark = pytest.mark.gpu

MATS = [fsg.MAT_AIR, fsg.MAT_SAND, fsg.MAT_WATER, fsg.MAT_STONE]


def noise(rng, shape):
    """Records that differ from their neighbours in every byte they can."""
    rgba = rng.integers(0, 2**32, shape, dtype=np.uint64)
    temp = rng.integers(0, 2**16, shape, dtype=np.uint64)
    return rng.choice(np.array(MATS, np.uint64), shape) | temp << np.uint64(16) | rgba << np.uint64(32)


def patterns(rng, shape):
    base = noise(rng, shape)
    flat = np.full(shape, base[0, 0])
    cols = np.broadcast_to(base[:1], shape).copy()               # every row the one above
    runs = np.repeat(base[:, ::16], 16, axis=1)[:, :shape[1]]    # runs of records
    some = base.copy()
    some[rng.random(shape) < 0.5] = base[0, 0]
    rare = base.copy()
    rare[5::37] = base[4, 7]                                     # a row that is one run between noisy ones
    last = base.copy()
    last[-1] = base[0, 0]
    first = base.copy()
    first[0] = base[0, 0]
    byte = cols ^ (rng.integers(0, 2, shape, dtype=np.uint64) << np.uint64(40))  # one byte differs here and there
    moved = runs | (rng.integers(0, 2, shape, dtype=np.uint64) << np.uint64(8))
    return dict(noise=base, flat=flat, cols=cols, runs=runs, some=some, rare=rare, last=last, first=first, byte=byte,
                moved=moved)


@pytest.mark.parametrize("name", list(patterns(np.random.default_rng(0), (8, 16))))
@pytest.mark.parametrize("aux", ["none", "noise", "same"])
def test_row_patterns(ctx, orc, name, aux):
    rng = np.random.default_rng(12)
    print("pack rows", name, aux, flush=True)
    cells = patterns(rng, (128, 256))[name]
    l2 = None if aux == "none" else noise(rng, (128, 256)) if aux == "noise" else cells.copy()
    bg = None if aux == "none" else (noise(rng, (128, 256)) if aux == "noise" else cells) >> np.uint64(32)
    bg = None if bg is None else bg.astype(np.uint32)
    with fsg.World(ctx, 256, 128, 1, orc.default_config()) as w:
        w.upload(cells)
        got = w.pack(0, 0, 2, 1, layer2=l2, background=bg)
        w.upload(np.zeros_like(cells))
        st, _ph, l2b, bgb = w.unpack(0, 0, 2, 1, got, want_layer2=True, want_background=True)
        back = w.download()
    ref = oracle_images(orc, cells, 0, 0, 2, 1, None, l2, bg)
    for k in range(2):
        assert got[k] == ref[k], k
    assert (st == 0).all() and np.array_equal(back, cells)
    assert l2 is None or np.array_equal(l2b, l2)
    assert bg is None or np.array_equal(bgb, bg)


def one_value_rows(rng, shape):
    """Rows of one value, that of the record before them, which are not parsed."""
    base = noise(rng, shape)
    after = base.copy()
    after[1::3] = base[0:-1:3, -1:][:after[1::3].shape[0]]   # behind rows that end in literals
    pairs = base.copy()
    pairs[3::5] = pairs[4::5] = base[2:-1:5, -1:][:pairs[4::5].shape[0]]  # two in a row, then literals again
    most = np.full(shape, base[0, 0])
    most[40, 17:19] = base[1, :2]                            # one row of many with something in it
    ends = np.full(shape, base[0, 0])
    ends[0, 0] = base[1, 1]                                  # the block's first record
    ends[-1, -1] = base[2, 2]                                # and its last one
    return dict(after=after, pairs=pairs, most=most, ends=ends)


@pytest.mark.parametrize("name", ["after", "pairs", "most", "ends"])
@pytest.mark.parametrize("aux", ["none", "same"])
def test_rows_of_one_value(ctx, orc, name, aux):
    print("pack rows of one value", name, aux, flush=True)
    cells = one_value_rows(np.random.default_rng(5), (128, 128))[name]
    cells = np.concatenate([cells, one_value_rows(np.random.default_rng(6), (128, 128))[name]], axis=1)
    l2 = None if aux == "none" else cells.copy()
    bg = None if aux == "none" else (cells >> np.uint64(32)).astype(np.uint32)
    with fsg.World(ctx, 256, 128, 1, orc.default_config()) as w:
        w.upload(cells)
        got = w.pack(0, 0, 2, 1, layer2=l2, background=bg)
        w.upload(np.zeros_like(cells))
        st, _ph, l2b, bgb = w.unpack(0, 0, 2, 1, got, want_layer2=True, want_background=True)
        back = w.download()
    assert got == oracle_images(orc, cells, 0, 0, 2, 1, None, l2, bg)
    assert (st == 0).all() and np.array_equal(back, cells)
    assert l2 is None or (np.array_equal(l2b, l2) and np.array_equal(bgb, bg))
