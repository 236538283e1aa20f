"""The decode of few blocks, a workgroup each, against the oracle's decoder:
raw blocks in calls small enough to take it (a call of one block, and slices
of the blocks the one-wave decode is tested with, corrupt ones too), long
literal runs and matches, and offsets across its batches; nothing is written
past a block's capacity.  A call of more blocks gives the same."""
import ctypes as C

import numpy as np
import pytest

import falling_sand_engine_amd as fsg
import lz4ref
from test_pack import O, corrupt_cases, far_match_blocks, host_decoder, lz4_seq, sample_blocks, short_sequence_blocks


def long_blocks():
    """Sequences at the lines of a batch: as many length bytes as it takes and
    one more, outputs of its size and one more, offsets over its history."""
    rng = np.random.default_rng(4)
    out = []
    for n_lit, ml in ((15 + 255 * 7, 19 + 255 * 7), (15 + 255 * 8, 19 + 255 * 8), (8188, 4), (8189, 4), (16000, 9000),
                      (1, 8191), (1, 70000), (20000, 5)):
        for off in (1, 12, 4096, 8192, 8193, 16384, 65535):
            dec_len, blk = 0, b""
            for k in range(4):
                lit = rng.integers(0, 256, n_lit + k).astype(np.uint8).tobytes()
                dec_len += len(lit)
                blk += lz4_seq(lit, min(off, dec_len), ml + k)
                dec_len += ml + k
            for k in range(40):  # short ones after long ones
                blk += lz4_seq(bytes([k] * (k % 9)), min(off, dec_len), 4 + k)
                dec_len += k % 9 + 4 + k
            blk += lz4_seq(rng.integers(0, 256, 13).astype(np.uint8).tobytes())
            out.append((blk, dec_len + 13))
    return out


def all_cases(corrupt):
    blocks = sample_blocks(lz4ref.lib() is not None) + far_match_blocks() + short_sequence_blocks()
    return blocks + long_blocks() + corrupt_cases(blocks, corrupt, 31)


def test_wide_decoder_matches_oracle_on_the_host():
    f = host_decoder().fsg_test_lz4_decode_wide
    f.restype, f.argtypes = C.c_int, [C.c_void_p, C.c_int, C.c_void_p, C.c_int]
    for src, cap in all_cases(1200):
        s = np.frombuffer(src, np.uint8) if src else np.zeros(1, np.uint8)
        want = O.lz4_decode(src, cap)
        out = np.full(cap + 64, 0xA5, np.uint8)
        r = f(s.ctypes.data, len(src), out.ctypes.data, cap)
        assert (out[:cap].tobytes() if r == cap else None) == want, (len(src), cap, r)
        assert (out[cap:] == 0xA5).all()


@pytest.mark.gpu
@pytest.mark.parametrize("per_call", [1, 61, 700])
def test_wide_decoder_matches_oracle_on_the_device(ctx, orc, per_call):
    cases = all_cases(900)
    if per_call == 1:
        cases = cases[::29]
    for a in range(0, len(cases), per_call):
        print("wide decode", a, per_call, flush=True)
        part = cases[a:a + per_call]
        for k, ((src, cap), (r, out)) in enumerate(zip(part, fsg.lz4_decode_blocks(ctx, part, guard=64))):
            want = orc.lz4_decode(src, cap)
            assert (out[:cap] if r == cap else None) == want, (a + k, len(src), cap, r)
            assert out[cap:] == b"\xa5" * 64, a + k


@pytest.mark.gpu
@pytest.mark.parametrize("cx,cy", [(16, 16), (20, 20), (32, 24), (40, 20)])  # up to two blocks per CU, six, more
@pytest.mark.parametrize("features", ["none", "few", "one chunk", "one bad"])
def test_unpack_of_nearly_empty_chunks(ctx, cx, cy, features):
    """Between two and six blocks per compute unit the longest input decides
    between a wave and a workgroup per block: chunks of air, with scattered
    cells, with one chunk of noise among them, and with one image cut short."""
    W, H = 128 * cx, 128 * cy
    rng = np.random.default_rng(cx)
    cells = np.zeros((H, W), np.uint64)
    noise = (rng.integers(0, 8, (H, W)).astype(np.uint64) | (rng.integers(0, 2**32, (H, W), dtype=np.uint64) << np.uint64(32)))
    if features == "few":
        at = rng.random((H, W)) < 0.01
        cells[at] = noise[at]
    elif features != "none":
        cells[256:384, 128:256] = noise[256:384, 128:256]
    print(f"unpack {cx}x{cy} {features}", flush=True)
    with fsg.World(ctx, W, H, 1) as w:
        w.upload(cells)
        images = w.pack(0, 0, cx, cy)
        w.generate(2, 3)
        want = cells
        if features == "one bad":
            images[2 * cx + 1] = images[2 * cx + 1][:-1]
            want = cells.copy()
            want[256:384, 128:256] = w.download()[256:384, 128:256]
        status = w.unpack(0, 0, cx, cy, images)[0]
        assert [k for k, s in enumerate(status) if s] == ([2 * cx + 1] if features == "one bad" else [])
        assert np.array_equal(w.download(), want)
