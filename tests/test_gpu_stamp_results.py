"""Stamp results counted and listed on the device: bodies whose pixels lie in
any order and with gaps, displaced lists cut at every kind of capacity (none,
shorter and longer than a workgroup's share, past the size that comes with the
counts), per-body hits, and bodies that overlap refused."""
import numpy as np
import pytest

import falling_sand_engine_amd as fsg
from bodies import random_bodies

pytestmark = pytest.mark.gpu


def shuffled(rng, bodies, pixels):
    """The same bodies with their pixel blocks in another order and unused
    pixels between them."""
    order = rng.permutation(len(bodies))
    out, blocks, off = [None] * len(bodies), [], 0
    for b in order:
        B = bodies[b]
        n = B.mat_w * B.mat_h
        gap = int(rng.integers(0, 3)) * 7
        blocks.append(np.full(gap, fsg.make_cell(fsg.MAT_STONE, 100), np.uint64))
        blocks.append(pixels[B.pixel_offset:B.pixel_offset + n])
        off += gap
        out[b] = fsg.Body(B.pos_x_q16, B.pos_y_q16, B.cos_q16, B.sin_q16, B.mat_w, B.mat_h, off, B.enabled)
        off += n
    return out, np.concatenate(blocks)


@pytest.mark.parametrize("nb,max_side,skip", [(1, 4, 0), (7, 20, 1), (60, 40, 0), (300, 12, 1)])
@pytest.mark.parametrize("cap", [0, 1, 255, 5000, 200000])
def test_results_match_oracle(ctx, orc, nb, max_side, skip, cap):
    W, H = 400, 300
    rng = np.random.default_rng(nb)
    cells = fsg.generate(2, W, H, nb)
    bodies, pixels = shuffled(rng, *random_bodies(rng, W, H, nb, max_side=max_side))
    cfg = orc.default_config(chunk_skip=skip)
    print(f"stamp results nb={nb} pixels={pixels.size} cap={cap} skip={skip}", flush=True)
    ref = cells.copy()
    rs = orc.stamp(ref, cfg, bodies, pixels, displaced_cap=cap)
    with fsg.World(ctx, W, H, 3, cfg) as w:
        w.upload(cells)
        gs = w.stamp_bodies(bodies, pixels, displaced_cap=cap)
        got = w.download()
        px = w.unstamp_bodies(pixels.size)
        back = w.download()
    assert np.array_equal(got, ref)
    live = sum(int(np.count_nonzero(pixels[B.pixel_offset:B.pixel_offset + B.mat_w * B.mat_h] & np.uint64(15)))
               for B in bodies if B.enabled)
    assert gs["unplaced"] == live - rs["placed"]
    for k in ("placed", "displaced", "hits_sand", "hits_soup", "displaced_cells"):
        assert gs[k] == rs[k], k
    ref_px = orc.unstamp(ref, cfg, bodies, pixels)
    assert np.array_equal(px, ref_px) and np.array_equal(back, ref)


def test_overlapping_bodies_refused(ctx):
    px = np.full(64, fsg.make_cell(fsg.MAT_STONE), np.uint64)
    ok = [fsg.body_from_pose(5, 5, 0, 4, 4, 32), fsg.body_from_pose(5, 5, 0, 4, 4, 16), fsg.body_from_pose(5, 5, 0, 4, 4, 48)]
    with fsg.World(ctx, 64, 64, 0) as w:
        for bad in ([fsg.body_from_pose(5, 5, 0, 4, 4, 47)], [fsg.body_from_pose(5, 5, 0, 4, 4, 49)],
                    [fsg.body_from_pose(5, 5, 0, 1, 1, 20)]):
            with pytest.raises(fsg.FsgError) as e:
                w.stamp_bodies(ok + bad, px)
            assert e.value.status == -1
        assert w.stamp_bodies(ok, px)["placed"] > 0
        w.unstamp_bodies(px.size)


@pytest.mark.parametrize("cap", [1000, 400000])
def test_displaced_list_of_many_workgroups(ctx, orc, cap):
    """Three bodies of 100,000 pixels over sand and water: 1,172 workgroups
    count them, in groups of 256."""
    W, H = 900, 700
    cells = np.full((H, W), fsg.make_cell(fsg.MAT_SAND, 320, 5), np.uint64)
    cells[:, ::3] = fsg.make_cell(fsg.MAT_AIR, 320, 0)
    cells[::7] = fsg.make_cell(fsg.MAT_WATER, 320, 6)
    rng = np.random.default_rng(1)
    px = np.full(300000, fsg.make_cell(fsg.MAT_STONE, 320, 7), np.uint64)
    px[rng.random(px.size) < 0.2] = 0
    px[100000:170000] = 0  # (workgroups and a whole group with none displaced)
    bodies = [fsg.body_from_pose(250 + 180 * k, 200 + 150 * k, 0.3 * k, 400, 250, 100000 * k) for k in range(3)]
    cfg = orc.default_config()
    print(f"stamp 300,000 pixels cap={cap}", flush=True)
    ref = cells.copy()
    rs = orc.stamp(ref, cfg, bodies, px, displaced_cap=cap)
    with fsg.World(ctx, W, H, 3, cfg) as w:
        w.upload(cells)
        gs = w.stamp_bodies(bodies, px, displaced_cap=cap)
        assert np.array_equal(w.download(), ref)
    assert rs["displaced"] > 65536 and len(gs["displaced_cells"]) == min(cap, rs["displaced"])
    for k in ("placed", "displaced", "hits_sand", "hits_soup", "displaced_cells"):
        assert gs[k] == rs[k], k
