// fsg_lz4_wide.hpp -- LZ4 block decoding by a workgroup, for few blocks.
//
// One wave decodes a block (fsg_lz4.hpp) as a chain of groups of at most 64
// output bytes, about 1300 cycles each; with fewer blocks than the chip has
// wave slots that chain is the whole time (256 chunks of 128 x 128, 17 MB of
// images: 3.4 ms).  Here a workgroup of WT threads
// takes a block by batches of up to WIN input and TOUT output bytes (two input
// bytes a thread; one: 1.29 ms for those 256 chunks, two 1.13; 512 threads with
// one: 1.85):
//   1. every input byte of the batch is parsed as if a sequence began there
//      (length, literals, offset, match, where the next one begins);
//   2. the positions each 64-byte segment is left at are found for every
//      entry by pointer jumping, the segments' real entries by following
//      those, and the real sequences of a segment from its entry;
//   3. a prefix sum gives each sequence its output position, and a bitmap of
//      those positions gives each output byte its sequence;
//   4. an output byte is a literal, a byte written before the batch, or a copy
//      of an earlier byte of the batch: those are pointers, followed with
//      their progress written back, so chains of matches halve at each step.
// A sequence that the batch's limits leave out (near the block's ends, more
// than 8 length bytes, an offset that is 0 or reaches before the output)
// is decoded alone by the whole workgroup with the rules of decode_block; the
// rules hold for the others because they end 16 bytes before either end.
//
// G is the group policy: each(f) runs f(t) for the threads this one stands
// for (itself on the device, all WT in turn on the host), sync() is the
// workgroup barrier, Reg<T> holds one value per thread; chain(), prefix(), waves_before()
// (the sum of earlier waves' numbers, and of all) and cover() (words [a, b) of
// each thread set to its value) work on the 64 threads of a wave.
#pragma once
#include "fsg_lz4.hpp"

namespace fsg_lz4 {

constexpr int WT = 1024;           // threads
constexpr int CAND = 2;            // input positions parsed by a thread per batch
constexpr int WIN = CAND * WT;     // and by all: position c * WT + t is thread t's c-th
constexpr int IBUF = 16 * WT;      // block bytes in LDS
constexpr int TOUT = 8192;         // output bytes per batch at most
constexpr int ORING = 8192;        // the last output bytes in LDS
constexpr int MAXSEQ = WIN / 3 + 2; // sequences of a batch (each takes 3 bytes or more)
constexpr int MAXEXT = 8;          // length bytes of a batched sequence
constexpr uint32_t STOP = 0x8000u; // no sequence is parsed at this position
constexpr uint64_t RESOLVED = 0x8000800080008000ull;

struct WideLds {
    uint8_t in[IBUF];          // block bytes [ib, ib + IBUF), 16-byte aligned
    uint64_t P[TOUT / 4 + 1];  // 16 bits per output byte: 0x8000 | byte, or the entry it copies
    uint32_t ring[ORING / 4];  // output byte q at byte (q + dst % 4) % ORING
    uint32_t H[TOUT / 32];     // bit: a sequence's output starts
    int last[TOUT / 32 + 1];   // the last sequence starting before each word of H
    uint32_t sa[MAXSEQ], sb[MAXSEQ];          // start | literals << 16; literals' place in `in` | offset << 16
    uint16_t leave[WIN];       // where the chain from this position leaves its segment
    uint32_t wcount[WIN / 64], wout[WIN / 64];
    uint32_t cut;              // start << 11 | position of the first sequence left out
};

// m mod o for 0 <= m < 2^20, o > 0 (the quotient's estimate is off by at most one).
__host__ __device__ inline int mod_small(int m, int o) {
#ifdef __HIP_DEVICE_COMPILE__
    const float inv = __builtin_amdgcn_rcpf((float)o);
#else
    const float inv = 1.0f / (float)o;
#endif
    int r = m - (int)((float)m * inv) * o;
    r = r < 0 ? r + o : r;
    return r >= o ? r - o : r;
}

template <class G>
__host__ __device__ inline int decode_wide(const uint8_t *src, int n, uint8_t *dst, int cap, WideLds &S, G &g) {
    if (n <= 0 || cap < 0) return -1;
    if (cap == 0) return (n == 1 && src[0] == 0) ? 0 : -1;
    uint8_t *const ring = reinterpret_cast<uint8_t *>(S.ring);
    const int adst = (int)((uintptr_t)dst & 3);
    int ip = 0, op = 0, ib = 0;
    bool loaded = false;
    typename G::template Reg<uint32_t> nx[CAND];
    typename G::template Reg<int> ll[CAND], lp[CAND], off[CAND], len[CAND], entry[CAND], before[CAND];
    typename G::template Reg<uint64_t> mask[CAND];
    for (;;) {
        if (ip >= n) return -1;
        if (!loaded || (ib + IBUF < n && ip + IBUF / 4 > ib + IBUF)) {
            ib = ip - (int)((uintptr_t)(src + ip) & 15);
            loaded = true;
            g.each([&](int t) {
                const int a = ib + 16 * t;
                if (a >= 0 && a + 16 <= n) {
                    *reinterpret_cast<uint4 *>(S.in + 16 * t) = *reinterpret_cast<const uint4 *>(src + a);
                } else {
                    for (int k = 0; k < 16; k++) S.in[16 * t + k] = (a + k >= 0 && a + k < n) ? src[a + k] : 0;
                }
            });
            g.sync();
        }
        // 1. candidates; every byte read lies in [ip, lim), inside the buffer
        const int lim = n - 16 < ib + IBUF ? n - 16 : ib + IBUF;
        g.each([&](int t) {
            for (int c = 0; c < CAND; c++) {
                const int p = ip + c * WT + t;
                auto b = [&](int i) { return (uint32_t)S.in[i - ib]; };
                uint32_t to = STOP;
                int l = 0, m = 0, q = p + 1, o = 0, e = 0;
                auto more = [&](int &v, int &at) -> bool {  // length bytes; false: too many, or past lim
                    uint32_t s = 255;
                    for (int k = 0; k < MAXEXT && s == 255; k++) {
                        if (at >= lim) return false;
                        s = b(at++);
                        v += (int)s;
                    }
                    return s != 255;
                };
                if (p < lim) {
                    const uint32_t token = b(p);
                    l = (int)(token >> 4);
                    m = (int)(token & 15u);
                    if (l != RUN_MASK || more(l, q)) {
                        e = q + l;
                        if (e + 2 <= lim) {
                            o = (int)(b(e) | b(e + 1) << 8);
                            int r = e + 2;
                            if ((m != 15 || more(m, r)) && r <= lim) to = (uint32_t)(r - ip);
                        }
                    }
                }
                nx[c][t] = to;
                ll[c][t] = l;
                lp[c][t] = q - ib;
                off[c][t] = o;
                len[c][t] = l + m + MINMATCH;
                S.leave[c * WT + t] = (uint16_t)(to == STOP ? STOP | (uint32_t)(c * WT + t) : to);
            }
            if (t < TOUT / 32) S.H[t] = 0;
            if (t == 0) {
                S.cut = ~0u;
                S.last[0] = -1;
            }
        });
        g.sync();
        // 2. each position's way out of its segment (a step more is 3 bytes on
        // or more; others' progress, read in any order, only shortens it)
        g.each([&](int t) {
            for (int c = 0; c < CAND; c++) {
                const int at = c * WT + t;
                const uint32_t end = (uint32_t)(at | 63) + 1;
                uint32_t e = S.leave[at];
                while (e < end) {  // STOP lies above every position
                    e = S.leave[e];
                    S.leave[at] = (uint16_t)e;
                }
            }
        });
        g.sync();
        uint32_t last = 0;  // where the real chain ends: past the batch, or STOP | position
        g.each([&](int t) {
            uint32_t e = 0;
            for (int c = 0; c < CAND; c++) {
                const uint32_t seg = (uint32_t)(c * WT + (t & ~63));
                while (e < seg) e = g.uniform(S.leave[e]);
                entry[c][t] = e < seg + 64 ? (int)(e - seg) : -1;
            }
            while (e < (uint32_t)WIN) e = g.uniform(S.leave[e]);
            last = e;
        });
        for (int c = 0; c < CAND; c++) g.chain(nx[c], entry[c], mask[c], c * WT);
        // 3. output positions
        for (int c = 0; c < CAND; c++)
            g.prefix([&](int t) { return (mask[c][t] >> (t & 63)) & 1u ? len[c][t] : 0; }, before[c],
                     S.wout + c * (WT / 64));
        g.each([&](int t) {
            if ((t & 63) == 0)
                for (int c = 0; c < CAND; c++) S.wcount[c * (WT / 64) + (t >> 6)] = (uint32_t)popc64(mask[c][t]);
        });
        g.sync();
        int total = 0;
        g.each([&](int t) {
            for (int c = 0; c < CAND; c++) {
                int none;
                const int at = before[c][t] + g.waves_before(t, c, S.wout, total), end = at + len[c][t];
                const bool in = (mask[c][t] >> (t & 63)) & 1u, fits = end <= TOUT;
                const int r = g.waves_before(t, c, S.wcount, none) +
                              popc64(mask[c][t] & ((1ull << (t & 63)) - 1));
                // (a sequence after the cut stands past the batch's last byte)
                g.cover(t, S.last, r, (at >> 5) + 1, in && fits ? (end >> 5) + 1 : 0);
                if (!in) continue;
                if (off[c][t] == 0 || off[c][t] > op + at + ll[c][t] || !fits || op + end + 16 > cap)
                    g.min(&S.cut, (uint32_t)(at < 2 * TOUT ? at : 2 * TOUT) << 11 | (uint32_t)(c * WT + t));
                if (!fits) continue;
                S.sa[r] = (uint32_t)at | (uint32_t)ll[c][t] << 16;
                S.sb[r] = (uint32_t)lp[c][t] | (uint32_t)off[c][t] << 16;
                g.or_(&S.H[at >> 5], 1u << (at & 31));
            }
        });
        g.sync();
        const uint32_t cut = g.uniform(S.cut);
        const int T = cut == ~0u ? total : (int)(cut >> 11);
        const int next = cut != ~0u ? (int)(cut & 2047u) : last >= STOP ? (int)(last & ~STOP) : (int)last;
        if (T == 0) {
            // one sequence by decode_block's rules, read through `byte` and
            // copied by all threads; its sources are in the output itself
            auto byte = [&](int i) -> int { return i >= ib && i < ib + IBUF ? S.in[i - ib] : src[i]; };
            int k = ip;
            const int token = byte(k++);
            int l = token >> 4;
            if (l == RUN_MASK) {
                const int end = n - RUN_MASK;
                if (k >= end) return -1;
                int s;
                do {
                    s = byte(k++);
                    l += s;
                    if (k > end || l > cap) return -1;
                } while (s == 255);
            }
            auto put = [&](int q, uint8_t v, bool recent) {
                dst[q] = v;
                if (recent) ring[(q + adst) & (ORING - 1)] = v;
            };
            const int at = k, cpy = op + l;
            const bool tail = cpy > cap - MFLIMIT || at + l > n - (2 + 1 + LASTLITERALS);
            if (tail && (at + l != n || cpy > cap)) return -1;
            g.each([&](int t) {
                for (int j = t; j < l; j += WT) put(op + j, src[at + j], j >= l - ORING);
            });
            if (tail) return cpy;
            op = cpy;
            k += l;
            const int o = byte(k) | byte(k + 1) << 8;
            k += 2;
            int m = token & 15;
            if (m == 15) {
                const int end = n - LASTLITERALS + 1;
                int s;
                do {
                    s = byte(k++);
                    m += s;
                    if (k > end || m > cap) return -1;
                } while (s == 255);
            }
            m += MINMATCH;
            if (o > op) return -1;
            if (op + m > cap - LASTLITERALS) return -1;
            g.sync();
            g.each([&](int t) {
                for (int j = t; j < m; j += WT)
                    put(op + j, o ? dst[op - o + (o < m ? j % o : j)] : (uint8_t)0, j >= m - ORING);
            });
            op += m;
            ip = k;
            g.sync();
            continue;
        }
        // 4. output bytes, a thread per aligned word of the output; entry i of P
        // is output byte i - a0 of the batch
        const int a0 = (adst + op) & 3, words = (T + a0 + 3) >> 2;
        g.each([&](int t) {
            for (int w = t; w < words; w += WT) {
                const int j0 = 4 * w - a0;
                uint64_t four = 0;
                for (int u = 0; u < 4; u++) {
                    const int j = j0 + u < 0 ? 0 : j0 + u < T ? j0 + u : T - 1;  // past either end: any byte's
                    const uint32_t upto = S.H[j >> 5] & (~0u >> (31 - (j & 31)));
                    const int q = S.last[j >> 5] + __builtin_popcount(upto);
                    const uint32_t a = S.sa[q], bb = S.sb[q];
                    const int l = (int)(a >> 16), rel = j - (int)(a & 0xFFFFu), m = rel - l, o = (int)(bb >> 16);
                    // j - m - o + (m mod o), before the match
                    const int from = m < o ? j - o : j - m - o + mod_small(m, o);
                    const int back = op + from + adst;
                    const uint8_t *p = rel < l ? S.in + (int)(bb & 0xFFFFu) + rel : ring + (back & (ORING - 1));
                    uint32_t v = *p;
                    if (rel >= l && from < -ORING) v = dst[op + from];
                    v = rel >= l && from >= 0 ? (uint32_t)(from + a0) : v | 0x8000u;
                    four |= (uint64_t)v << (16 * u);
                }
                S.P[w] = four;
            }
        });
        g.sync();
        g.each([&](int t) {
            const uint16_t *P = reinterpret_cast<const uint16_t *>(S.P);
            for (int w = t; w < words; w += WT) {
                const int j0 = 4 * w - a0;
                uint64_t four = S.P[w];
                while ((four & RESOLVED) != RESOLVED) {
                    uint64_t to = 0;
                    for (int u = 0; u < 4; u++) {
                        const uint32_t e = (uint32_t)(four >> (16 * u)) & 0xFFFFu;
                        const uint32_t x = P[(e & 0x8000u) ? (uint32_t)(4 * w + u) : e];
                        to |= (uint64_t)((e & 0x8000u) ? e : x) << (16 * u);
                    }
                    four = to;
                    S.P[w] = four;
                }
                const uint32_t v = (uint32_t)(four & 0xFFu) | (uint32_t)(four >> 8 & 0xFF00u) |
                                   (uint32_t)(four >> 16 & 0xFF0000u) | (uint32_t)(four >> 24 & 0xFF000000u);
                if (j0 >= 0 && j0 + 4 <= T) {
                    *reinterpret_cast<uint32_t *>(dst + op + j0) = v;
                    S.ring[((op + j0 + adst) & (ORING - 1)) >> 2] = v;
                } else {
                    for (int u = 0; u < 4; u++)
                        if (j0 + u >= 0 && j0 + u < T) {
                            dst[op + j0 + u] = (uint8_t)(v >> (8 * u));
                            ring[(op + j0 + u + adst) & (ORING - 1)] = (uint8_t)(v >> (8 * u));
                        }
                }
            }
        });
        op += T;
        ip += next;
        g.sync();
    }
}

}  // namespace fsg_lz4
