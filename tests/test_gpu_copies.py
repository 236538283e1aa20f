"""Copies between the host and the device: rectangles of every width class
(whole rows, narrow, one row, one column), sizes on both sides of the staging
limit, and more uploads in flight than the staging holds."""
import numpy as np
import pytest

import falling_sand_engine_amd as fsg

pytestmark = pytest.mark.gpu


def cells_of(W, H, seed):
    rng = np.random.default_rng(seed)
    return (rng.integers(0, 8, (H, W)).astype(np.uint64) | (np.uint64(320) << np.uint64(16)) |
            (rng.integers(0, 2**32, (H, W), dtype=np.uint64) << np.uint64(32)))


@pytest.mark.parametrize("W,H", [(1, 1), (65, 33), (512, 256), (513, 256), (1024, 700)])  # 512 x 256: the limit
def test_rectangles(ctx, W, H):
    cells = cells_of(W, H, W)
    with fsg.World(ctx, W, H, 0) as w:
        w.upload(cells)
        w.render()
        layer = w.layer(fsg.LAYER_CELLS)
        for x0, y0, rw, rh in [(0, 0, W, H), (0, H // 2, W, 1), (W // 2, 0, 1, H), (W // 3, H // 3, W - W // 3, H - H // 3),
                               (0, 0, max(W - 1, 1), H), (W - 1, H - 1, 1, 1)]:
            assert np.array_equal(w.download(x0, y0, rw, rh), cells[y0:y0 + rh, x0:x0 + rw]), (x0, y0, rw, rh)
            assert np.array_equal(w.layer(fsg.LAYER_CELLS, x0, y0, rw, rh), layer[y0:y0 + rh, x0:x0 + rw])


@pytest.mark.parametrize("n", [1, 1000, 30000, 90000])  # 90,000 edits: past the limit
def test_uploads_in_flight(ctx, n):
    """Edit batches behind a long tick queue, each staged and the caller's
    arrays gone before the device reads them."""
    W = H = 512
    ref = cells_of(W, H, 5)
    rng = np.random.default_rng(n)
    with fsg.World(ctx, W, H, 0, fsg.default_config(reactions=0, temp_every=0)) as w, \
            fsg.World(ctx, W, H, 0) as busy:
        w.upload(ref)
        for k in range(8):
            busy.tick(50)
            busy.generate(2, k)  # an upload nobody waits for
            at = rng.choice(W * H, n, replace=False)
            vals = cells_of(1, n, k).ravel()
            arr = (fsg._abi.CellEdit * n)()
            a = np.frombuffer(arr, np.dtype([("x", np.int32), ("y", np.int32), ("c", np.uint64)]))
            a["x"], a["y"], a["c"] = at % W, at // W, vals
            fsg.check(fsg.lib().fsg_world_set_cells(w.handle, arr, n))
            ref.ravel()[at] = vals
        assert np.array_equal(w.download(), ref)


def test_rectangles_without_device_memory(ctx):
    """A download of part of a world succeeds when no device memory can be had
    for it."""
    W, H = 300, 200
    cells = cells_of(W, H, 3)
    with fsg.World(ctx, W, H, 0) as w:
        w.upload(cells)
        w.render()
        layer = w.layer(fsg.LAYER_CELLS)
        for x0, y0, rw, rh in [(0, 0, 299, 200), (17, 50, 200, 120), (299, 0, 1, 200)]:
            print(f"rectangle {x0},{y0} {rw}x{rh} without device memory", flush=True)
            try:
                ctx.inject_alloc_failures(1)
                assert np.array_equal(w.download(x0, y0, rw, rh), cells[y0:y0 + rh, x0:x0 + rw])
                ctx.inject_alloc_failures(1)
                assert np.array_equal(w.layer(fsg.LAYER_CELLS, x0, y0, rw, rh), layer[y0:y0 + rh, x0:x0 + rw])
            finally:
                ctx.inject_alloc_failures(0)


@pytest.mark.parametrize("rw,rh", [(4095, 2049), (4095, 4096), (2047, 4096)])  # bands of 2,048 and 4,098 rows
def test_rectangles_of_several_bands(ctx, rw, rh):
    W = H = 4096
    cells = cells_of(W, H, 4)
    with fsg.World(ctx, W, H, 0) as w:
        w.upload(cells)
        print(f"rectangle {rw}x{rh}", flush=True)
        assert np.array_equal(w.download(1, H - rh, rw, rh), cells[H - rh:, 1:1 + rw])


def test_copies_without_pinned_memory():
    """Small uploads and downloads succeed when the pinned staging cannot be
    had, and use it once it can."""
    W, H = 200, 100
    cells = cells_of(W, H, 6)
    cfg = fsg.default_config()
    cfg.n_materials = 9  # no class tables, whose upload would take the staging at creation
    cfg.materials[8] = cfg.materials[fsg.MAT_STONE]
    ps = [fsg.make_particle(fsg.make_cell(fsg.MAT_SAND, 320, i), 5.0 + i % 90, 5.0, 0.0, 0.0) for i in range(20000)]
    with fsg.Context(0) as c, fsg.World(c, W, H, 0, cfg) as w:
        w.upload(cells)
        w.particles_add(ps)  # 1.1 MB each: past the staging's size
        w.particles_add(ps[:19000])  # (and the list grows to 40,000)
        for fails in (1, 0):
            print(f"staging fails={fails}", flush=True)
            c.inject_alloc_failures(fails)
            w.particles_add(ps[:10])  # staged up; the list has room
            c.inject_alloc_failures(fails)
            assert np.array_equal(w.download(), cells)
            c.inject_alloc_failures(0)
        got = w.particles()
        assert [(p.x, p.tile.rgba) for p in got] == [(p.x, p.tile.rgba) for p in ps + ps[:19000] + ps[:10] + ps[:10]]
