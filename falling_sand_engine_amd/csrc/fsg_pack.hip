// fsg_pack.hip -- chunk .pack images made and read on the device.
//
// A .pack image (chunk.cpp:219-330 ChunkWrite, read back by chunk.cpp:74-217
// ChunkRead) holds one 128x128 chunk:
//   i8 generation phase, i32 src_size (393216), i32 compressed_size,
//   i32 src_size2 (65536), i32 compressed_size2,
//   LZ4 block of the 12-byte MaterialInstanceData records {u32 material
//   index, u32 colour, i16 temperature, 2 pad bytes} of tiles[] then layer2[],
//   LZ4 block of the u32 background.
// A record's index is the file's material index of the cell's material id
// (the world's pack map; by default the id itself), its colour and
// temperature are the cell's, and the cell's MOVED flag travels in bit 0 of
// pad byte 10, which ChunkRead ignores; so an image round-trips a chunk
// exactly, and every index it holds is a material the reader knows.
//
// Encoding: one workgroup per chunk and block.  The reference asks LZ4 for a
// hash-chain search (LZ4_compress_fast, acceleration 10); any parse of the
// block format decodes the same, so the encoder uses one that parallelises:
// every byte is compared with the byte one record back and one record row
// (128 records) back, runs of equal bytes of 4 or more become matches with
// that offset, and the rest are literals.  A wave parses one record row;
// matches do not cross rows, literal runs do (a prefix scan over the rows
// gives each row the literals carried into it).  Runs of identical cells,
// identical rows, and the fields that repeat between neighbouring records
// (material, temperature, alpha, padding) all become matches.  The last 12
// bytes of a block are literals, as the format requires.
//
// Decoding: one wave per block (fsg_lz4.hpp), four waves per workgroup, or for
// few blocks with enough input a workgroup each (fsg_lz4_wide.hpp), into a
// record staging area;
// then one workgroup per chunk checks every record and
// writes the cells.
#include "fsg_internal.hpp"
#include "fsg_lz4.hpp"
#include "fsg_lz4_wide.hpp"

#include <algorithm>
#include <cstring>

namespace {

constexpr int CW = FSG_CHUNK;                   // chunk side (const.h:19-20)
constexpr int RA = 12, RB = 4;                  // record sizes of the two blocks
constexpr int NA = CW * CW * 2 * RA;            // tiles + layer2 records: 393216
constexpr int NB = CW * CW * RB;                // background: 65536
constexpr int bound(int n) { return n + n / 255 + 16; }  // LZ4_compressBound (lz4.h)
constexpr int CAPA = bound(NA), CAPB = bound(NB);
constexpr size_t SLOT = ((size_t)CAPA + CAPB + 255) & ~(size_t)255;  // encoder output per chunk
constexpr size_t RAW = (size_t)NA + NB;          // decoder output per chunk
constexpr int HDR = 17;
constexpr int PT = 1024;                         // encoder threads

struct PackSrc {
    const uint64_t *cells;  // world grid
    int W;
    const uint64_t *l2;     // region layer2 cells, row width rw (null: empty)
    const uint32_t *bg;     // region background (null: 0)
    int rw, x0, y0, ncx;
    uint64_t keep;          // cell bits a record carries: ~0x1FF, plus MOVED unless FSG_PACK_NO_MOVED
    uint8_t to_file[16];    // file index of each material id
};

// A cell in record form: the material id replaced by its file index (< 256,
// bits 0-7) and MOVED kept or dropped (bit 8); temperature and colour as
// stored.  Record bytes are then plain bytes of this word (rbyte).
__device__ __forceinline__ uint64_t rec_form(const PackSrc &s, uint64_t v) {
    return (v & s.keep) | s.to_file[v & 15u];
}

// Record i of block A (tiles rows 0..127, then layer2) or B of chunk (cx, cy).
__device__ __forceinline__ uint64_t rec_a(const PackSrc &s, int cx, int cy, int i) {
    const int row = (i >> 7) & (CW - 1), col = i & (CW - 1);
    if (i < CW * CW) return rec_form(s, s.cells[(size_t)(s.y0 + cy * CW + row) * s.W + (s.x0 + cx * CW + col)]);
    return rec_form(s, s.l2 ? s.l2[(size_t)(cy * CW + row) * s.rw + cx * CW + col] : 0ull);
}
__device__ __forceinline__ uint64_t rec_b(const PackSrc &s, int cx, int cy, int i) {
    const int row = i >> 7, col = i & (CW - 1);
    return s.bg ? s.bg[(size_t)(cy * CW + row) * s.rw + cx * CW + col] : 0u;
}

// Byte b of the record of record-form value v: material index (u32, < 256),
// colour (u32), temperature (i16), pad byte 10 (MOVED), pad byte 11 (0); for
// block B the u32 itself.
template <int R>
__device__ __forceinline__ uint32_t rbyte(uint64_t v, int b) {
    if (R == RB) return (uint32_t)(v >> (8 * b)) & 0xFFu;
    switch (b) {
    case 0: return (uint32_t)v & 0xFFu;
    case 4: case 5: case 6: case 7: return (uint32_t)(v >> (32 + 8 * (b - 4))) & 0xFFu;
    case 8: return (uint32_t)(v >> 16) & 0xFFu;
    case 9: return (uint32_t)(v >> 24) & 0xFFu;
    case 10: return (uint32_t)(v >> 8) & 0xFFu;
    default: return 0u;
    }
}

// Bit b set where byte b of two records is equal (x = their xor).
template <int R>
__device__ __forceinline__ uint32_t eqmask(uint64_t x) {
    uint32_t m = 0;
#pragma unroll
    for (int b = 0; b < R; b++) m |= (rbyte<R>(x, b) == 0u ? 1u : 0u) << b;
    return m;
}

__device__ __forceinline__ int extlen(int v) { return v >= 15 ? (v - 15) / 255 + 1 : 0; }

constexpr int ROWS = NA / (CW * RA);  // most record rows of a block: 256

// One record row parsed by a wave, two records (W bytes) a lane.  The lanes
// compare their bytes with the record before and the row above and keep the
// two answers as bit masks; runs of equal kind start where a mask changes, and
// a run's end, the last match before a lane and the next one after it are
// found by ballots.  Positions are bytes from the row's start.
template <int R>
struct RowParse {
    static constexpr int W = 2 * R, S = CW * R;
    uint32_t word[W / 4];      // the lane's bytes
    uint32_t lmask, start;     // bytes that equal the record before; run starts
    uint32_t match;            // starts of match runs (4 bytes or more, not literals)
    int next;                  // first run start past the lane
    int pe;                    // end of the last match that starts before the lane (-1: none)
    uint64_t lanes;            // lanes in which a match starts
    bool one;                  // the whole row is one match with the record before; nothing else is set

    // End of the run that starts at bit b of the lane.
    __device__ int end_of(int lane, int b) const {
        const uint32_t m = start & ~((2u << b) - 1u);
        return m ? lane * W + __builtin_ctz(m) : next;
    }
    template <class Rec>
    __device__ void parse(int row, int lane, int n, const Rec &rec) {
        constexpr uint32_t FULL = (1u << W) - 1u;
        const int i = row * CW + 2 * lane;
        const uint64_t v0 = rec(i), v1 = rec(i + 1);
        const uint64_t u0 = row ? rec(i - CW) : 0ull, u1 = row ? rec(i + 1 - CW) : 0ull;
        uint64_t left = __shfl_up(v1, 1, 64);
        const uint64_t wrap = __shfl(u1, 63, 64);  // the row above's last record comes before this row's first
        if (lane == 0) left = wrap;
        one = row > 0 && (row + 1) * S <= n - fsg_lz4::MFLIMIT && !__ballot(((v1 ^ v0) | (v0 ^ left)) != 0);
        if (one) return;
        uint32_t mL = eqmask<R>(v1 ^ v0) << R, mU = 0;
        if (i > 0) mL |= eqmask<R>(v0 ^ left);
        if (row) mU = eqmask<R>(v0 ^ u0) | eqmask<R>(v1 ^ u1) << R;
        const int p0 = i * R, forced = n - fsg_lz4::MFLIMIT;  // bytes from forced on are literals
        const uint32_t live = p0 + W <= forced ? FULL : p0 >= forced ? 0u : (1u << (forced - p0)) - 1u;
        lmask = mL & live;
        const uint32_t umask = mU & ~mL & live;
        const uint32_t before = __shfl_up(((lmask >> (W - 1)) & 1u) | ((umask >> (W - 1)) & 1u) << 1, 1, 64);
        start = ((lmask ^ (lmask << 1 | (before & 1u))) | (umask ^ (umask << 1 | (before >> 1 & 1u)))) & FULL;
        if (lane == 0) start |= 1u;
        const uint64_t any = __ballot(start != 0), above = any & ~((2ull << lane) - 1ull);
        const int first = lane * W + (start ? __builtin_ctz(start) : 0);
        const int nf = __shfl(first, above ? __builtin_ctzll(above) : 0, 64);
        next = above ? nf : S;
        match = 0;
        int lme = 0;
        for (uint32_t m = start & (lmask | umask); m; m &= m - 1) {
            const int b = __builtin_ctz(m), e = end_of(lane, b);
            if (e - (lane * W + b) < fsg_lz4::MINMATCH) continue;
            match |= 1u << b;
            lme = e;
        }
        lanes = __ballot(match != 0);
        const uint64_t below = lanes & ((1ull << lane) - 1ull);
        const int pl = __shfl(lme, below ? 63 - __builtin_clzll(below) : 0, 64);
        pe = below ? pl : -1;
        auto put = [&](int k, uint64_t v) {
            if (R == RB) {
                word[k] = (uint32_t)v;
            } else {
                word[3 * k] = (uint32_t)v & 0xFFu;
                word[3 * k + 1] = (uint32_t)(v >> 32);
                word[3 * k + 2] = ((uint32_t)v >> 16) | ((uint32_t)v & 0xFF00u) << 8;
            }
        };
        put(0, v0);
        put(1, v1);
    }
    // Bytes of the lane's sequences; the row's first one without its literals
    // and their length bytes.
    __device__ int size(int lane) const {
        int sum = 0, prev = pe;
        for (uint32_t m = match; m; m &= m - 1) {
            const int b = __builtin_ctz(m), at = lane * W + b, e = end_of(lane, b), ll = prev < 0 ? 0 : at - prev;
            sum += 3 + extlen(ll) + ll + extlen(e - at - fsg_lz4::MINMATCH);
            prev = e;
        }
        return sum;
    }
    __device__ uint32_t byte(int b) const {
        uint32_t w = word[0];
#pragma unroll
        for (int k = 1; k < W / 4; k++) w = (b >> 2) == k ? word[k] : w;
        return w >> (8 * (b & 3)) & 0xFFu;
    }
};

// Output of one block: every store is checked against the block's capacity
// (the size pass keeps the writes inside it; the check keeps a slot's
// neighbours safe whatever happens).
struct Out {
    uint8_t *p;
    int cap;
    __device__ void put(int at, uint32_t v) const {
        if (at >= 0 && at < cap) p[at] = (uint8_t)v;
    }
};

__device__ __forceinline__ int put_len(const Out &o, int oc, int v) {
    if (v >= 15) {
        v -= 15;
        while (v >= 255) {
            o.put(oc++, 255);
            v -= 255;
        }
        o.put(oc++, (uint32_t)v);
    }
    return oc;
}

// Sums over the wave's lanes up to and with this one.
__device__ __forceinline__ int wave_sum(int v, int lane) {
    for (int d = 1; d < 64; d <<= 1) {
        const int o = __shfl_up(v, d, 64);
        v += lane >= d ? o : 0;
    }
    return v;
}

// Exclusive sums over the rows; every thread of the workgroup calls it.
__device__ __forceinline__ int rows_before(int v, int *sums, int *total) {
    const int t = threadIdx.x, lane = t & 63;
    const int s = wave_sum(v, lane);
    if (lane == 63 && t < ROWS) sums[t >> 6] = s;
    __syncthreads();
    int b = 0, all = 0;
    for (int w = 0; w < ROWS / 64; w++) {
        b += w < (t >> 6) ? sums[w] : 0;
        all += sums[w];
    }
    *total = all;
    __syncthreads();
    return b + s - v;
}

// A workgroup of PT threads encodes a block: its waves take the record rows in
// turn, first for the rows' sizes, then to write them.  Bound by the VALU work of
// the run loops, whose trips are the lane's with the most runs, and of a row's
// fixed part, which rows of one value do without.  (A thread per row walking its
// records: 1326 us for 256 basin chunks, so 191, for 2304 1577 and 893; for 256
// chunks of air 197 and 51, for 2304 881 and 459, 1282 with every row parsed.)
template <int R, class Rec>
__device__ void encode_block(int n, const Rec &rec, uint8_t *out, int cap, int32_t *size_out) {
    constexpr int S = CW * R, NW = PT / 64;
    const int rows = n / S, L = rows - 1, t = threadIdx.x, lane = t & 63, wv = t >> 6;
    __shared__ int hm[ROWS], lead[ROWS], trail[ROWS], rest[ROWS], carry[ROWS], start[ROWS], nxt[ROWS], sums[ROWS / 64];
    __shared__ int psum[ROWS + 1];
    __shared__ uint64_t has[ROWS / 64];
    __shared__ uint8_t one[ROWS];  // rows that are one match: sized without a parse, and not read again
    for (int r = wv; r < rows; r += NW) {
        RowParse<R> p;
        p.parse(r, lane, n, rec);
        if (lane == 0) one[r] = p.one;
        if (p.one) {
            if (lane == 0) {
                hm[r] = 1;
                lead[r] = trail[r] = 0;
                rest[r] = 3 + extlen(S - fsg_lz4::MINMATCH);
            }
            continue;
        }
        const int sum = wave_sum(p.size(lane), lane);
        const uint64_t lanes = p.lanes;
        // the row's first match, and the end of its last one
        int b = p.match ? lane * RowParse<R>::W + __builtin_ctz(p.match) : 0;
        int e = p.match ? p.end_of(lane, 31 - __builtin_clz(p.match)) : 0;
        b = __shfl(b, lanes ? __builtin_ctzll(lanes) : 0, 64);
        e = __shfl(e, lanes ? 63 - __builtin_clzll(lanes) : 0, 64);
        if (lane == 63) {
            hm[r] = lanes != 0;
            lead[r] = lanes ? b : S;
            trail[r] = lanes ? S - e : S;
            rest[r] = sum;
        }
    }
    __syncthreads();
    const bool mine = t < rows;
    int total;
    const int ps = rows_before(mine ? trail[t] : 0, sums, &total);
    const uint64_t hb = __ballot(mine && hm[t]);
    if (t < ROWS) {
        psum[t] = ps;
        if (lane == 0) has[wv] = hb;
    }
    __syncthreads();
    int sz = 0;
    if (mine) {
        // the literals carried into a row: the trailing ones since the last row with a match
        int prev = 0, nx = L;
        for (int w = t >> 6; w >= 0; w--) {
            const uint64_t m = w == (t >> 6) ? has[w] & ((1ull << lane) - 1ull) : has[w];
            if (m) {
                prev = 64 * w + 63 - __builtin_clzll(m);
                break;
            }
        }
        for (int w = t >> 6; w < ROWS / 64; w++) {
            const uint64_t m = w == (t >> 6) ? has[w] & ~((2ull << lane) - 1ull) : has[w];
            if (m) {
                nx = 64 * w + __builtin_ctzll(m);
                break;
            }
        }
        const int c = ps - psum[prev];
        carry[t] = c;
        nxt[t] = nx;
        if (hm[t]) sz = rest[t] + extlen(c + lead[t]) + c + lead[t];
        if (t == L) {
            const int llf = hm[t] ? trail[t] : c + S;
            sz += 1 + extlen(llf) + llf;
        }
    }
    const int at0 = rows_before(sz, sums, &total);
    if (mine) start[t] = at0;
    __syncthreads();
    if (total > cap) {  // cannot happen for these parses (sizes stay under the LZ4 bound)
        if (t == 0) *size_out = -1;
        return;
    }
    const Out o{out, cap};
    for (int r = wv; r < rows; r += NW) {
        if (one[r]) {
            if (lane == 0) {
                constexpr int ml = S - fsg_lz4::MINMATCH;
                o.put(start[r], (uint32_t)(min(carry[r], 15) << 4 | min(ml, 15)));
                int oc = put_len(o, start[r] + 1, carry[r]) + carry[r];
                o.put(oc++, (uint32_t)R);
                o.put(oc++, 0u);
                put_len(o, oc, ml);
            }
            continue;
        }
        RowParse<R> p;
        p.parse(r, lane, n, rec);
        constexpr int W = RowParse<R>::W;
        const int sum = wave_sum(p.size(lane), lane), rowsum = __shfl(sum, 63, 64);
        const int ll1 = carry[r] + lead[r], skip = extlen(ll1) + ll1;  // the first sequence's literals
        // where the row's trailing literals go: byte b of the row to tail + b
        int tail;
        if (r == L) {
            const int llf = hm[r] ? trail[r] : carry[r] + S;
            int oc = start[r] + (hm[r] ? rowsum + skip : 0);
            if (lane == 0) {
                o.put(oc, (uint32_t)(min(llf, 15) << 4));
                put_len(o, oc + 1, llf);
            }
            oc += 1 + extlen(llf);
            tail = oc + (llf - trail[r]) - (S - trail[r]);
        } else {
            const int u = nxt[r], ll0 = carry[u] + lead[u];
            tail = start[u] + 1 + extlen(ll0) + carry[u] + (r - u) * S;
        }
        // the lane's sequences, and where each one's literals go
        int oc = start[r] + (sum - p.size(lane)) + (p.pe < 0 ? 0 : skip);
        auto base_of = [&](int prev, int at) { return prev < 0 ? oc + 1 + extlen(ll1) + carry[r]
                                                               : oc + 1 + extlen(at - prev) - prev; };
        // the literals past the lane's last match belong to the next lane with one
        const int fb = p.match ? base_of(p.pe, lane * W + __builtin_ctz(p.match)) : 0;
        const uint64_t above = p.lanes & ~((2ull << lane) - 1ull);
        const int nb = __shfl(fb, above ? __builtin_ctzll(above) : 0, 64);
        int prev = p.pe, from = max(p.pe - lane * W, 0);
        auto literals = [&](int a, int b, int base) {
            for (int k = a; k < b; k++) o.put(base + lane * W + k, p.byte(k));
        };
        for (uint32_t m = p.match; m; m &= m - 1) {
            const int b = __builtin_ctz(m), at = lane * W + b, e = p.end_of(lane, b);
            const int ll = prev < 0 ? ll1 : at - prev, ml = e - at - fsg_lz4::MINMATCH;
            literals(from, b, base_of(prev, at));
            o.put(oc, (uint32_t)(min(ll, 15) << 4 | min(ml, 15)));
            oc = put_len(o, oc + 1, ll) + ll;
            const int off = (p.lmask >> b & 1u) ? R : S;
            o.put(oc++, (uint32_t)off & 0xFFu);
            o.put(oc++, (uint32_t)off >> 8);
            oc = put_len(o, oc, ml);
            prev = e;
            from = e - lane * W;
        }
        literals(from, W, above ? nb : tail);
    }
    if (t == 0) *size_out = total;
}

struct RecA {
    PackSrc s;
    int cx, cy;
    __device__ uint64_t operator()(int i) const { return rec_a(s, cx, cy, i); }
};
struct RecB {
    PackSrc s;
    int cx, cy;
    __device__ uint64_t operator()(int i) const { return rec_b(s, cx, cy, i); }
};

// grid: x = chunk, y = block (0: tiles + layer2, 1: background)
__global__ __launch_bounds__(PT) void k_pack_encode(PackSrc s, uint8_t *slots, int32_t *sizes) {
    const int c = blockIdx.x, cx = c % s.ncx, cy = c / s.ncx;
    uint8_t *slot = slots + (size_t)c * SLOT;
    if (blockIdx.y == 0) encode_block<RA>(NA, RecA{s, cx, cy}, slot, CAPA, &sizes[2 * c]);
    else encode_block<RB>(NB, RecB{s, cx, cy}, slot + CAPA, CAPB, &sizes[2 * c + 1]);
}

// Image offsets (exclusive scan of 17 + A + B over the chunks); off[n] = total,
// or -1 when a block failed.  One workgroup.
__global__ __launch_bounds__(1024) void k_pack_offsets(const int32_t *sizes, int n, int64_t *off) {
    __shared__ int64_t part[16];
    __shared__ int bad;
    const int t = threadIdx.x, per = (n + 1023) / 1024, a = min(n, t * per), b = min(n, a + per);
    if (t == 0) bad = 0;
    __syncthreads();
    int64_t s = 0;
    for (int c = a; c < b; c++) {
        if (sizes[2 * c] < 0 || sizes[2 * c + 1] < 0) bad = 1;
        s += HDR + sizes[2 * c] + sizes[2 * c + 1];
    }
    int64_t sum = s;
    for (int d = 1; d < 64; d <<= 1) {
        const int64_t v = __shfl_up(sum, d, 64);
        sum += (t & 63) >= d ? v : 0;
    }
    if ((t & 63) == 63) part[t >> 6] = sum;
    __syncthreads();
    int64_t o = sum - s, all = 0;
    for (int w = 0; w < 16; w++) {
        o += w < (t >> 6) ? part[w] : 0;
        all += part[w];
    }
    if (t == 0) off[n] = bad ? -1 : all;
    for (int c = a; c < b; c++) {
        off[c] = o;
        o += HDR + sizes[2 * c] + sizes[2 * c + 1];
    }
}

__device__ __forceinline__ void put_i32(uint8_t *p, int32_t v) {
    for (int k = 0; k < 4; k++) p[k] = (uint8_t)((uint32_t)v >> (8 * k));
}

// Thread t of nt copies its share of len bytes: aligned words of the
// destination, each from the two aligned words of the source it lies in (the
// word past the last byte is read: encoder slots have room behind them).
__device__ __forceinline__ void copy_words(uint8_t *dst, const uint8_t *src, int len, int t, int nt) {
    const int head = min(len, (int)(-(uintptr_t)dst & 3)), words = (len - head) >> 2, done = head + 4 * words;
    if (t < head) dst[t] = src[t];
    if (t < len - done) dst[done + t] = src[done + t];
    const int sh = (int)((uintptr_t)(src + head) & 3);
    const uint32_t *p = reinterpret_cast<const uint32_t *>(src + head - sh);
    uint32_t *q = reinterpret_cast<uint32_t *>(dst + head);
    for (int k = t; k < words; k += nt)
        q[k] = (uint32_t)((((uint64_t)p[k + 1] << 32) | p[k]) >> (8 * sh));
}
static_assert(SLOT >= (size_t)CAPA + CAPB + 8, "room behind block B's last byte");

// Writes each chunk's image: header, then block A, then block B.  ASM workgroups
// a chunk (of bytes by one workgroup a chunk: 107 us for 256 chunks, 17 MB; so
// 8.7).
constexpr int ASM = 8;
__global__ __launch_bounds__(256) void k_pack_assemble(const uint8_t *slots, const int32_t *sizes,
                                                       const int64_t *off, const int8_t *phase, uint8_t *img) {
    const int c = blockIdx.x, t = (int)(blockIdx.y * 256 + threadIdx.x);
    if (off[gridDim.x] < 0) return;
    const int a = sizes[2 * c], b = sizes[2 * c + 1];
    uint8_t *o = img + off[c];
    const uint8_t *sa = slots + (size_t)c * SLOT, *sb = sa + CAPA;
    if (t == 0) {
        o[0] = (uint8_t)phase[c];
        put_i32(o + 1, NA);
        put_i32(o + 5, a);
        put_i32(o + 9, NB);
        put_i32(o + 13, b);
    }
    copy_words(o + HDR, sa, a, t, 256 * ASM);
    copy_words(o + HDR + a, sb, b, t, 256 * ASM);
}

// Decoder input: per block, its bytes in[off, off + n) (n < 0: no block, the
// result is -1) and its output out[dst, dst + cap).
struct DecDesc {
    int64_t off, dst;
    int32_t n, cap;
};

// The match table of the decode kernel (LDS, filled by each workgroup before
// its waves decode; read only after that).
__shared__ uint8_t dec_modtab[fsg_lz4::MODTAB];

// The lane policy of the decode kernel: this thread's own lane.  A wave's
// window and ring are its own and a wave's LDS accesses execute in order, so
// ordering the lanes' accesses needs only wavefront-scope fences around a
// wave barrier (which keeps the compiler from moving accesses across it); a
// workgroup barrier would tie the workgroup's waves together and also wait
// for every outstanding output store.
struct WaveLane {
    int lane;
    template <class F>
    __device__ void each(F f) const {
        f(lane);
    }
    __device__ void barrier() const {
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    }
    __device__ uint32_t uniform(uint32_t x) const { return __builtin_amdgcn_readfirstlane(x); }
    __device__ uint32_t lane_value(uint32_t v, int k, const uint8_t *) const {
        return (uint32_t)__builtin_amdgcn_readlane((int)v, k);
    }
    __device__ uint32_t own(uint32_t v, int, const uint8_t *) const { return v; }
    __device__ uint32_t mod(int i) const { return dec_modtab[i]; }
    // lane vectors are the lane's own register; called with every lane active
    using V = uint32_t;
    template <class F>
    __device__ V make(F f) const {
        return f(lane);
    }
    __device__ uint32_t get(V v, int) const { return v; }
    __device__ uint32_t lane_of(V v, int k) const { return (uint32_t)__builtin_amdgcn_readlane((int)v, k); }
    __device__ uint64_t ballot(V v) const { return __builtin_amdgcn_ballot_w64(v != 0u); }
    __device__ V shfl(V v, V i) const { return (uint32_t)__builtin_amdgcn_ds_bpermute((int)(i << 2), (int)v); }
    __device__ uint32_t below(uint64_t m, int) const {
        return __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u));
    }
};

// One wave per block, four blocks per workgroup (a workgroup per wave would
// leave CUs short of waves: their workgroup slots run out first).  Wave
// v = blockIdx.x * 4 + wave takes block desc[v]; the unpack lists every
// chunk's tiles-and-layer2 block (384 KiB decoded) before the background
// blocks (64 KiB), so a workgroup holds blocks of one kind and its waves end
// together (a mixed one stays resident until its long blocks end), and the
// long blocks start first.  Each wave keeps its own block window and output
// ring in LDS and decodes alone (no workgroup barrier); result[v] is the
// decoded size, or -1 for a block lz4.c rejects.  A 2 KB ring (this
// encoder's offsets are at most one record row, 1536 bytes) keeps the LDS at
// 16.6 KB per workgroup, so 8 waves per SIMD fit (58 VGPRs): unpack 14.6 ->
// 13.9 ms on 16384 chunks against a 4 KB ring at 6 waves.
constexpr int DW = 4;  // waves (blocks) per decode workgroup

__global__ __launch_bounds__(64 * DW) __attribute__((amdgpu_waves_per_eu(8))) void k_pack_decode(
    const uint8_t *in, const DecDesc *desc, uint8_t *out, int32_t *result, int nblocks) {
    __shared__ __align__(16) uint8_t win[DW][fsg_lz4::IW];
    __shared__ uint8_t ring[DW][fsg_lz4::RING];
    __shared__ uint32_t gdesc[DW][fsg_lz4::GMAX];
    for (int i = threadIdx.x; i < fsg_lz4::MODTAB; i += 64 * DW) dec_modtab[i] = fsg_lz4::modtab_entry(i);
    __syncthreads();
    // the wave's index as a uniform, so that the block's descriptor and the
    // whole parse (positions, lengths, limits) live in scalar registers
    const int wv = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)), lane = threadIdx.x & 63;
    const int v = blockIdx.x * DW + wv;
    if (v >= nblocks) return;
    const DecDesc d = desc[v];
    int r = -1;
    if (d.n >= 0) {
        fsg_lz4::Staged<WaveLane> M{in + d.off, d.n, out + d.dst, win[wv], ring[wv], gdesc[wv], -(1 << 30),
                                    WaveLane{lane}, 0u, 0};
        r = fsg_lz4::decode_block(d.n, d.cap, M);
    }
    if (lane == 0) result[v] = r;
}

// The group policy of the wide decode: this thread.
struct WideGroup {
    int t;
    template <class T>
    struct Reg {
        T v;
        __device__ T &operator[](int) { return v; }
    };
    template <class F>
    __device__ void each(F f) {
        f(t);
    }
    __device__ void sync() { __syncthreads(); }
    __device__ uint32_t uniform(uint32_t x) { return (uint32_t)__builtin_amdgcn_readfirstlane((int)x); }
    __device__ void min(uint32_t *p, uint32_t v) { atomicMin(p, v); }
    __device__ void or_(uint32_t *p, uint32_t v) { atomicOr(p, v); }
    // the sequences on the chain from the wave's entry
    __device__ void chain(Reg<uint32_t> &nx, Reg<int> &entry, Reg<uint64_t> &mask, int base) {
        const int seg = __builtin_amdgcn_readfirstlane(t & ~63) + base;
        uint64_t m = 0;
        for (int at = __builtin_amdgcn_readfirstlane(entry.v); at >= 0 && at < 64;) {
            const uint32_t to = (uint32_t)__builtin_amdgcn_readlane((int)nx.v, at);
            if (to == fsg_lz4::STOP) break;
            m |= 1ull << at;
            at = (int)to - seg;
        }
        mask.v = m;
    }
    // the wave's running sum, along rows of 16 lanes, then across them
    __device__ int inclusive(int v) {
        v += __builtin_amdgcn_update_dpp(0, v, 0x111, 0xF, 0xF, true);   // row_shr:1
        v += __builtin_amdgcn_update_dpp(0, v, 0x112, 0xF, 0xF, true);   // row_shr:2
        v += __builtin_amdgcn_update_dpp(0, v, 0x114, 0xF, 0xF, true);   // row_shr:4
        v += __builtin_amdgcn_update_dpp(0, v, 0x118, 0xF, 0xF, true);   // row_shr:8
        v += __builtin_amdgcn_update_dpp(0, v, 0x142, 0xA, 0xF, false);  // row_bcast:15 into rows 1 and 3
        v += __builtin_amdgcn_update_dpp(0, v, 0x143, 0xC, 0xF, false);  // row_bcast:31 into rows 2 and 3
        return v;
    }
    template <class F>
    __device__ void prefix(F f, Reg<int> &before, uint32_t *sums) {
        const int v = f(t), s = inclusive(v);
        before.v = s - v;
        if ((t & 63) == 63) sums[t >> 6] = (uint32_t)s;
    }
    __device__ int waves_before(int, int c, const uint32_t *sums, int &total) {
        constexpr int NW = fsg_lz4::WIN / 64;
        const int s = inclusive((t & 63) < NW ? (int)sums[t & 63] : 0);
        const int wv = __builtin_amdgcn_readfirstlane(t >> 6) + c * (fsg_lz4::WT / 64);
        total = __builtin_amdgcn_readlane(s, NW - 1);
        return wv ? __builtin_amdgcn_readlane(s, wv - 1) : 0;
    }
    // a thread's word where it has one, the wave's threads for more
    __device__ void cover(int, int *p, int v, int a, int b) {
        if (b - a == 1) p[a] = v;
        for (uint64_t m = __ballot(b - a > 1); m; m &= m - 1) {
            const int k = __builtin_ctzll(m);
            const int kv = __builtin_amdgcn_readlane(v, k), ka = __builtin_amdgcn_readlane(a, k),
                      kb = __builtin_amdgcn_readlane(b, k);
            for (int w = ka + (t & 63); w < kb; w += 64) p[w] = kv;
        }
    }
};

// A workgroup per block (fsg_lz4_wide.hpp): a third of the time is the output
// bytes' lookups (VALU issue), a sixth the barriers, the rest LDS latency of the
// parse and the chains.
__global__ __launch_bounds__(fsg_lz4::WT) void k_pack_decode_wide(const uint8_t *in, const DecDesc *desc, uint8_t *out,
                                                                  int32_t *result) {
    __shared__ __align__(16) fsg_lz4::WideLds S;
    const DecDesc d = desc[blockIdx.x];
    WideGroup g{(int)threadIdx.x};
    int r = -1;
    if (d.n >= 0) r = fsg_lz4::decode_wide(in + d.off, d.n, out + d.dst, d.cap, S, g);
    if (threadIdx.x == 0) result[blockIdx.x] = r;
}

// A workgroup per block or a wave per block.  By waves a call takes what its
// longest block takes, by its input bytes mostly; by workgroups, of which two
// are resident on a compute unit, it grows with the blocks past that, as a
// workgroup does more work for a block than a wave.  So up to two blocks per
// compute unit it is workgroups, and up to six if the longest block's input is
// long enough for the number of blocks.  us for
// chunk images (two blocks each, half of them short), waves / workgroups: 1
// chunk 3233 / 925, 256 3535 / 947, 400 3527 / 1599, 576 3522 / 2425, 768 3513
// / 2577 (1024: 3.8 / 4.1 ms a call); nearly empty ones, of 3,003 bytes, 1 853
// / 498, 256 876 / 595, 400 877 / 1019, 768 884 / 1732; 400 of 4.6 KB 976 /
// 1053, of 7.9 KB 1168 / 1064; 576 of 7.7 KB 1163 / 1583, of 15.5 KB 1642 /
// 1555; 768 of 15.5 KB 1636 / 1775, of 39 KB 2909 / 1728.  (Raw blocks as small
// as 1,000 bytes, 512 of them, take 7 to 34 by waves and 14 to 43 so, which is
// lost in such a call's copies; 1,500 go by waves.)
bool decode_wide_pays(const fsg_ctx *c, const std::vector<DecDesc> &desc) {
    const int64_t n = (int64_t)desc.size(), cu = c->n_cu;
    if (n <= 2 * cu || n > 6 * cu) return n <= 2 * cu;
    int32_t longest = 0;
    for (const DecDesc &d : desc) longest = std::max(longest, d.n);
    return longest * cu >= (n - 2 * cu) * 5120;
}

// desc: the blocks as d_desc has them.
void launch_decode(const fsg_ctx *c, const uint8_t *in, const std::vector<DecDesc> &desc, const DecDesc *d_desc,
                   uint8_t *out, int32_t *result) {
    const unsigned n = (unsigned)desc.size();
    if (decode_wide_pays(c, desc))
        k_pack_decode_wide<<<n, fsg_lz4::WT, 0, c->stream>>>(in, d_desc, out, result);
    else
        k_pack_decode<<<(n + DW - 1) / DW, 64 * DW, 0, c->stream>>>(in, d_desc, out, result, (int)n);
}

// Little-endian u32 at a 4-byte aligned staging address (records are 12 or
// 4 bytes and each chunk's staging starts at a multiple of 4).
__device__ __forceinline__ uint32_t ld32(const uint8_t *p) { return *reinterpret_cast<const uint32_t *>(p); }
static_assert(RAW % 4 == 0 && NA % 4 == 0 && RA % 4 == 0 && RB % 4 == 0, "aligned record words");

struct UnpackDst {
    uint64_t *cells;  // world grid
    int W, x0, y0, ncx, rw;
    uint64_t *l2;     // region layer2 out (null: not kept)
    uint32_t *bg;     // region background out (null: not kept)
    uint32_t moved;   // MOVED taken from pad byte 10 (else clear)
    int n;            // chunks: status[c] and status[n + c] are chunk c's decoded block sizes
    int16_t from_file[256];  // material id of each file index, or -1
};

// One workgroup per chunk: records -> cells, after checking every material
// index against the map (a bad one fails the chunk and leaves its cells as
// they were).
__global__ __launch_bounds__(256) void k_pack_cells(const uint8_t *raw, const int32_t *status, UnpackDst d,
                                                    int32_t *chunk_status) {
    __shared__ int bad;
    const int c = blockIdx.x, t = threadIdx.x, cx = c % d.ncx, cy = c / d.ncx;
    if (status[c] != NA || status[d.n + c] != NB) {
        if (t == 0) chunk_status[c] = FSG_ERR_INVALID;
        return;
    }
    if (t == 0) bad = 0;
    __syncthreads();
    const uint8_t *r = raw + (size_t)c * RAW;
    int mybad = 0;
    for (int i = t; i < 2 * CW * CW; i += 256) {
        const uint32_t idx = ld32(r + (size_t)i * RA);
        mybad |= idx > 0xFFu || d.from_file[idx & 0xFFu] < 0;
    }
    if (mybad) bad = 1;
    __syncthreads();
    if (bad) {
        if (t == 0) chunk_status[c] = FSG_ERR_INVALID;
        return;
    }
    const int nrec = d.l2 ? 2 * CW * CW : CW * CW;  // layer2 records are read only when kept
    for (int i = t; i < nrec; i += 256) {
        const uint8_t *q = r + (size_t)i * RA;
        const uint32_t w2 = ld32(q + 8);  // temperature, pad byte 10, pad byte 11
        const uint64_t v = (uint64_t)(uint16_t)d.from_file[ld32(q)] | (d.moved ? (w2 >> 8) & 0x100u : 0u) |
                           ((uint64_t)(w2 & 0xFFFFu) << 16) | ((uint64_t)ld32(q + 4) << 32);
        const int row = (i >> 7) & (CW - 1), col = i & (CW - 1);
        if (i < CW * CW) d.cells[(size_t)(d.y0 + cy * CW + row) * d.W + (d.x0 + cx * CW + col)] = v;
        else if (d.l2) d.l2[(size_t)(cy * CW + row) * d.rw + cx * CW + col] = v;
    }
    if (d.bg)
        for (int i = t; i < CW * CW; i += 256)
            d.bg[(size_t)(cy * CW + (i >> 7)) * d.rw + cx * CW + (i & (CW - 1))] = ld32(r + NA + (size_t)i * RB);
    if (t == 0) chunk_status[c] = FSG_OK;
}

using fsg_impl::dev_alloc;
using fsg_impl::dev_free;

// Grows a world-owned device buffer to `bytes` (contents not kept).
int grow(fsg_ctx *c, void **p, size_t *cap, size_t bytes) {
    if (*cap >= bytes) return FSG_OK;
    dev_free(*p);
    *p = nullptr;
    *cap = 0;
    if (dev_alloc(c, p, bytes)) return FSG_ERR_NOMEM;
    *cap = bytes;
    return FSG_OK;
}

int region_ok(const fsg_world *w, int x0, int y0, int ncx, int ncy) {
    if (x0 < 0 || y0 < 0 || ncx <= 0 || ncy <= 0 || ncx > w->d.W / CW || ncy > w->d.H / CW) return 0;
    return (int64_t)x0 + (int64_t)ncx * CW <= w->d.W && (int64_t)y0 + (int64_t)ncy * CW <= w->d.H;
}

int32_t rd_i32(const uint8_t *p) {
    int32_t v;
    std::memcpy(&v, p, 4);
    return v;
}

void default_map(const fsg_config &cfg, fsg_pack_map *m) {
    std::memset(m, 0, sizeof(*m));
    for (int i = 0; i < 16; i++) m->to_file[i] = (uint32_t)i;
    for (int i = 0; i < 256; i++) m->from_file[i] = (int16_t)((uint32_t)i < cfg.n_materials ? i : -1);
}

// The map the world's pack calls use.
const fsg_pack_map &world_map(fsg_world *w) {
    if (!w->pack_map_set) default_map(w->cfg, &w->pack_map);
    return w->pack_map;
}

}  // namespace

extern "C" int fsg_pack_map_default(const fsg_config *cfg, fsg_pack_map *map) {
    if (!cfg || !map || cfg->n_materials > FSG_MAX_MATERIALS) return FSG_ERR_INVALID;
    default_map(*cfg, map);
    return FSG_OK;
}

extern "C" int fsg_world_set_pack_map(fsg_world *w, const fsg_pack_map *map) {
    if (!w) return FSG_ERR_INVALID;
    if (!map) {
        w->pack_map_set = false;
        return FSG_OK;
    }
    for (uint32_t m = 0; m < w->cfg.n_materials; m++)
        if (map->to_file[m] > 0xFFu) return FSG_ERR_INVALID;
    for (int i = 0; i < 256; i++)
        if (map->from_file[i] < -1 || map->from_file[i] >= (int)w->cfg.n_materials) return FSG_ERR_INVALID;
    if (map->flags & ~FSG_PACK_NO_MOVED) return FSG_ERR_INVALID;
    w->pack_map = *map;
    w->pack_map_set = true;
    return FSG_OK;
}

extern "C" int fsg_world_pack(fsg_world *w, int32_t x0, int32_t y0, int32_t ncx, int32_t ncy, const int8_t *phase,
                              const fsg_cell *layer2, const uint32_t *background, size_t *image_bytes) {
    if (!w || !image_bytes || !region_ok(w, x0, y0, ncx, ncy)) return FSG_ERR_INVALID;
    const size_t n = (size_t)ncx * ncy, rcells = n * CW * CW;
    if (layer2)  // layer2 records are cells of the world's materials too
        for (size_t i = 0; i < rcells; i++)
            if ((layer2[i].mat & 0xFE00u) || (uint32_t)(layer2[i].mat & 0xFFu) >= w->cfg.n_materials)
                return FSG_ERR_INVALID;
    fsg_ctx *c = w->ctx;
    HIPCHK(hipSetDevice(c->device));
    // per-chunk device state: encoder slots, images (worst case), sizes, offsets, phases;
    // the region's layer2 / background when given
    const size_t b_small = ((n * 8 + (n + 1) * 8 + n + 255) & ~(size_t)255);
    if (grow(c, &w->d_pack_slots, &w->pack_slots_cap, n * SLOT) ||
        grow(c, &w->d_pack_img, &w->pack_img_cap, n * (HDR + CAPA + CAPB)) ||
        grow(c, &w->d_pack_small, &w->pack_small_cap, b_small))
        return FSG_ERR_NOMEM;
    const size_t b_l2 = layer2 ? rcells * 8 : 0, b_bg = background ? rcells * 4 : 0;
    if (b_l2 + b_bg && grow(c, &w->d_pack_aux, &w->pack_aux_cap, b_l2 + b_bg)) return FSG_ERR_NOMEM;
    int32_t *d_sizes = static_cast<int32_t *>(w->d_pack_small);
    int64_t *d_off = reinterpret_cast<int64_t *>(d_sizes + 2 * n);
    int8_t *d_phase = reinterpret_cast<int8_t *>(d_off + n + 1);
    w->pack_phase.assign(n, 0);
    if (phase) std::copy(phase, phase + n, w->pack_phase.begin());
    if (int rc = fsg_impl::copy_in(c, d_phase, w->pack_phase.data(), n)) return rc;
    PackSrc s{};
    s.cells = w->d.buf[w->d.tick & 1];
    s.W = w->d.W;
    s.rw = ncx * CW;
    s.x0 = x0;
    s.y0 = y0;
    s.ncx = ncx;
    const fsg_pack_map &map = world_map(w);
    s.keep = (map.flags & FSG_PACK_NO_MOVED) ? ~0x1FFull : ~0xFFull;
    for (int m = 0; m < 16; m++) s.to_file[m] = (uint8_t)map.to_file[m];
    char *aux = static_cast<char *>(w->d_pack_aux);
    if (layer2) {
        HIPCHK(hipMemcpyAsync(aux, layer2, b_l2, hipMemcpyHostToDevice, c->stream));
        s.l2 = reinterpret_cast<const uint64_t *>(aux);
    }
    if (background) {
        HIPCHK(hipMemcpyAsync(aux + b_l2, background, b_bg, hipMemcpyHostToDevice, c->stream));
        s.bg = reinterpret_cast<const uint32_t *>(aux + b_l2);
    }
    uint8_t *slots = static_cast<uint8_t *>(w->d_pack_slots), *img = static_cast<uint8_t *>(w->d_pack_img);
    k_pack_encode<<<dim3((unsigned)n, 2), PT, 0, c->stream>>>(s, slots, d_sizes);
    k_pack_offsets<<<1, 1024, 0, c->stream>>>(d_sizes, (int)n, d_off);
    k_pack_assemble<<<dim3((unsigned)n, ASM), 256, 0, c->stream>>>(slots, d_sizes, d_off, d_phase, img);
    HIPCHK(hipGetLastError());
    w->pack_sizes.resize(2 * n);
    int64_t total = 0;
    if (int rc = fsg_impl::copy_out(c, {{w->pack_sizes.data(), d_sizes, 2 * n * 4}, {&total, d_off + n, 8}})) return rc;
    if (total < 0) {
        w->pack_n = 0;
        return FSG_ERR_DEVICE;
    }
    for (size_t k = 0; k < n; k++) image_bytes[k] = HDR + (size_t)w->pack_sizes[2 * k] + w->pack_sizes[2 * k + 1];
    w->pack_n = n;
    w->pack_total = (size_t)total;
    return FSG_OK;
}

extern "C" int fsg_world_pack_download(fsg_world *w, void *out, size_t cap) {
    if (!w || !out) return FSG_ERR_INVALID;
    if (w->pack_n == 0) return FSG_ERR_STATE;
    if (cap < w->pack_total) return FSG_ERR_INVALID;
    fsg_ctx *c = w->ctx;
    HIPCHK(hipSetDevice(c->device));
    return fsg_impl::copy_out(c, {{out, w->d_pack_img, w->pack_total}});
}

extern "C" int fsg_world_unpack(fsg_world *w, int32_t x0, int32_t y0, int32_t ncx, int32_t ncy, const void *images,
                                const size_t *image_bytes, int8_t *phase, fsg_cell *layer2, uint32_t *background,
                                int32_t *status) {
    if (!w || !status || !region_ok(w, x0, y0, ncx, ncy)) return FSG_ERR_INVALID;
    const size_t n = (size_t)ncx * ncy, rcells = n * CW * CW;
    if (images && !image_bytes) return FSG_ERR_INVALID;
    if (!images && w->pack_n != n) return FSG_ERR_STATE;  // the last pack's images, same chunk count
    fsg_ctx *c = w->ctx;
    HIPCHK(hipSetDevice(c->device));
    // descriptors of the 2n blocks from the headers (chunk.cpp:83-145)
    // chunk k's blocks: desc[k] (tiles and layer2, NA bytes) and desc[n + k] (background, NB)
    std::vector<DecDesc> desc(2 * n);
    std::vector<int8_t> ph(n, 0);
    const uint8_t *src = nullptr;
    size_t in_total = 0;
    if (images) {
        const uint8_t *p = static_cast<const uint8_t *>(images);
        for (size_t k = 0; k < n; k++) {
            const size_t len = image_bytes[k];
            DecDesc a{(int64_t)in_total + HDR, (int64_t)(k * RAW), -1, NA}, b{0, (int64_t)(k * RAW + NA), -1, NB};
            if (len >= (size_t)HDR) {
                ph[k] = (int8_t)p[in_total];
                const int32_t sa = rd_i32(p + in_total + 1), ca = rd_i32(p + in_total + 5);
                const int32_t sb = rd_i32(p + in_total + 9), cb = rd_i32(p + in_total + 13);
                if (sa == NA && sb == NB && ca >= 0 && cb >= 0 && (size_t)HDR + (size_t)ca + (size_t)cb <= len) {
                    a.n = ca;
                    b.off = a.off + ca;
                    b.n = cb;
                }
            }
            desc[k] = a;
            desc[n + k] = b;
            in_total += len;
        }
        if (grow(c, &w->d_pack_in, &w->pack_in_cap, std::max<size_t>(in_total, 1))) return FSG_ERR_NOMEM;
        src = static_cast<const uint8_t *>(w->d_pack_in);
    } else {
        int64_t o = 0;
        for (size_t k = 0; k < n; k++) {
            const int32_t ca = w->pack_sizes[2 * k], cb = w->pack_sizes[2 * k + 1];
            desc[k] = DecDesc{o + HDR, (int64_t)(k * RAW), ca, NA};
            desc[n + k] = DecDesc{o + HDR + ca, (int64_t)(k * RAW + NA), cb, NB};
            ph[k] = w->pack_phase[k];
            o += HDR + ca + cb;
        }
        src = static_cast<const uint8_t *>(w->d_pack_img);
    }
    const size_t b_desc = (2 * n * sizeof(DecDesc) + 255) & ~(size_t)255, b_st = (3 * n * 4 + 255) & ~(size_t)255;
    const size_t b_l2 = layer2 ? rcells * 8 : 0, b_bg = background ? rcells * 4 : 0;
    if (grow(c, &w->d_pack_raw, &w->pack_raw_cap, n * RAW) ||
        grow(c, &w->d_pack_dec, &w->pack_dec_cap, b_desc + b_st + b_l2 + b_bg))
        return FSG_ERR_NOMEM;
    if (images)  // the last thing that can fail for want of memory is behind it
        if (int rc = fsg_impl::copy_in(c, w->d_pack_in, images, in_total, true)) return rc;
    char *dec = static_cast<char *>(w->d_pack_dec);
    DecDesc *d_desc = reinterpret_cast<DecDesc *>(dec);
    int32_t *d_bst = reinterpret_cast<int32_t *>(dec + b_desc), *d_cst = d_bst + 2 * n;
    UnpackDst d{};
    d.cells = w->d.buf[w->d.tick & 1];
    d.W = w->d.W;
    d.x0 = x0;
    d.y0 = y0;
    d.ncx = ncx;
    d.rw = ncx * CW;
    d.l2 = layer2 ? reinterpret_cast<uint64_t *>(dec + b_desc + b_st) : nullptr;
    d.bg = background ? reinterpret_cast<uint32_t *>(dec + b_desc + b_st + b_l2) : nullptr;
    const fsg_pack_map &map = world_map(w);
    d.moved = (map.flags & FSG_PACK_NO_MOVED) ? 0u : 1u;
    d.n = (int)n;
    std::memcpy(d.from_file, map.from_file, sizeof(d.from_file));
    if (int rc = fsg_impl::copy_in(c, d_desc, desc.data(), 2 * n * sizeof(DecDesc))) return rc;
    if (b_l2 + b_bg) HIPCHK(hipMemsetAsync(dec + b_desc + b_st, 0, b_l2 + b_bg, c->stream));  // failed chunks: 0
    uint8_t *raw = static_cast<uint8_t *>(w->d_pack_raw);
    launch_decode(c, src, desc, d_desc, raw, d_bst);
    k_pack_cells<<<(unsigned)n, 256, 0, c->stream>>>(raw, d_bst, d, d_cst);
    HIPCHK(hipGetLastError());
    if (int rc = fsg_impl::copy_out(c, {{status, d_cst, n * 4},
                                        {layer2, d.l2, layer2 ? b_l2 : 0},
                                        {background, d.bg, background ? b_bg : 0}}))
        return rc;
    if (phase) std::copy(ph.begin(), ph.end(), phase);
    // new cells, as after fsg_world_upload
    w->d.force_tick = w->d.tick;
    w->stamped = false;
    w->prev_valid = false;
    return FSG_OK;
}

namespace {
struct DeviceBuffer {  // freed on every return path
    void *p = nullptr;
    ~DeviceBuffer() {
        if (p) (void)hipFree(p);
    }
};
}  // namespace

extern "C" int fsg_lz4_decode_blocks(fsg_ctx *c, const void *src, size_t src_len, const int64_t *src_off,
                                     const int32_t *src_bytes, const int32_t *cap, int32_t n, void *out,
                                     size_t out_len, const int64_t *out_off, int32_t *result) {
    if (!c || n < 0) return FSG_ERR_INVALID;
    if (n == 0) return FSG_OK;
    if (!src || !src_off || !src_bytes || !cap || !out || !out_off || !result) return FSG_ERR_INVALID;
    std::vector<DecDesc> desc((size_t)n);
    for (int32_t k = 0; k < n; k++) {
        if (src_off[k] < 0 || src_bytes[k] < 0 || (uint64_t)src_off[k] + (uint64_t)src_bytes[k] > src_len ||
            cap[k] < 0 || out_off[k] < 0 || (uint64_t)out_off[k] + (uint64_t)cap[k] > out_len)
            return FSG_ERR_INVALID;
        desc[k] = DecDesc{src_off[k], out_off[k], src_bytes[k], cap[k]};
    }
    HIPCHK(hipSetDevice(c->device));
    DeviceBuffer d_src, d_out, d_desc, d_res;
    HIPCHK(hipMalloc(&d_src.p, std::max<size_t>(src_len, 1)));
    HIPCHK(hipMalloc(&d_out.p, std::max<size_t>(out_len, 1)));
    HIPCHK(hipMalloc(&d_desc.p, (size_t)n * sizeof(DecDesc)));
    HIPCHK(hipMalloc(&d_res.p, (size_t)n * 4));
    if (src_len) HIPCHK(hipMemcpyAsync(d_src.p, src, src_len, hipMemcpyHostToDevice, c->stream));
    if (out_len) HIPCHK(hipMemcpyAsync(d_out.p, out, out_len, hipMemcpyHostToDevice, c->stream));
    HIPCHK(hipMemcpyAsync(d_desc.p, desc.data(), (size_t)n * sizeof(DecDesc), hipMemcpyHostToDevice, c->stream));
    launch_decode(c, static_cast<const uint8_t *>(d_src.p), desc, static_cast<const DecDesc *>(d_desc.p),
                  static_cast<uint8_t *>(d_out.p), static_cast<int32_t *>(d_res.p));
    HIPCHK(hipGetLastError());
    if (out_len) HIPCHK(hipMemcpyAsync(out, d_out.p, out_len, hipMemcpyDeviceToHost, c->stream));
    HIPCHK(hipMemcpyAsync(result, d_res.p, (size_t)n * 4, hipMemcpyDeviceToHost, c->stream));
    HIPCHK(hipStreamSynchronize(c->stream));
    return FSG_OK;
}
