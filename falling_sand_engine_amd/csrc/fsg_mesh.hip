// fsg_mesh.hip -- outlines of solid cells for the host physics engine:
// the marching-squares step of world::updateChunkMesh (world.cpp:722-895)
// and of updateRigidBodyHitbox (world.cpp:288-510), on the device.
//
// One workgroup per region (a 128x128 chunk of the grid, or an island's body
// image).  The region's mask, the reference's edge candidates (a set cell
// whose right, lower and lower-right neighbours are not all set, and whose
// marching-squares vertex value is not 15) and the edgeSeen marks are bit
// planes in LDS, built by all threads.  The reference walks candidates in
// row order, skipping the ones an earlier walk marked.  Here a wave takes the
// next 64 unmarked candidates at a time and every lane walks its own
// (FindPerimeter, physics_math.cpp:1881-1965), noting which candidates of the
// batch its walk marks; a scalar pass over the batch in row order then keeps
// the walks the reference would make.  A walk that meets an earlier candidate
// of its batch stops there: it is on that candidate's loop, which almost
// always marks it.  A candidate that is reached unmarked and whose walk
// stopped so, or for want of room (RUNS runs), has its walk finished by the
// whole wave, with the lanes sharing the marks and the farthest-point search,
// before the pass goes on; so the result never rests on a guess.  Meanwhile a
// second wave simplifies the last batch's loops, a loop per lane (Ramer-
// Douglas-Peucker, physics_math.cpp:1766-1812; f32 arithmetic as the reference
// does it, with no fused multiply-add, so its decisions are the reference's).
// Bound: the latency of the longest walk of each batch, an LDS read per step
// (of a plane of vertex values, which also flags the batch's candidates).
// Whole calls, against one walk at a time by one wave: every chunk of a 2048^2
// world with loose stone on a fifth of its cells (88,128 loops) 12.86 -> 0.73
// ms, of a 4096^2 world on half (428,601 loops, many of over 64 runs) 21.5 ->
// 10.0, of a 2048^2 basin world (54 long loops) 0.65 -> 0.36.
// Kept loops (3 or more vertices) are appended to output pools, one pair of
// atomics per batch, and put in region and trace order on the device.
#include "fsg_internal.hpp"

#include <algorithm>
#include <cstring>

namespace {

constexpr int MT = 256;                                 // threads per workgroup, one region
constexpr int MBITS = FSG_MESH_MAX_CELLS;               // mask bits per region
constexpr int MWORDS = MBITS / 32;
constexpr int MAXV = (128 + 1) * (128 + 1) + 2;         // runs of one loop of a 16384-cell region, bound
constexpr int LCAP = 1024;                              // loops up to this many runs stay in LDS
constexpr int RUNS = 64;                                // runs of a loop one lane walks (and bits of its keep mask)
constexpr int SECT = 32;                                // longest RDP section a lane of a whole-wave walk takes
constexpr int VCAP = MBITS + 256 + 64;                  // vertices of a region at most 255 cells wide and high
constexpr uint32_t LIVE = 0x80u;                        // vertex of a candidate of the batch

struct MeshSrc {
    const uint64_t *cells;  // region r's cell (x, y) is cells[off[r] + y * pitch[r] + x]
    uint32_t setmask;       // material ids whose cells are set (SOLID for the grid, not AIR for images)
};

struct MeshRegionDev {
    int64_t off;            // first cell
    int32_t pitch, w, h;
    uint32_t region;        // index in the caller's array
};

struct MeshOut {
    fsg_mesh_loop *loops;   // pool of loops (region, seq in first_loop order via `seq`)
    uint32_t *seq;          // per pooled loop: its trace order within its region
    uint32_t *voff;         // and the vertices of the region's loops before it
    uint32_t *verts;        // pool of vertices, (x | y << 16)
    uint32_t loop_cap, vert_cap;
    unsigned int *counters; // [0] loops, [1] vertices, [2] overflow, [3] walk failures
    uint32_t *scratch;      // per workgroup: MAXV vertices + MAXV stack entries
    uint32_t *regcnt;       // per caller's region: its loops (zero for regions not traced)
    uint32_t *regvert;      // and their vertices
};

__device__ __forceinline__ bool bit_at(const uint32_t *b, int i) { return (b[i >> 5] >> (i & 31)) & 1u; }

// isSet of vertex coordinates (x, y): cell (x - 1, y - 1) inside the region.
__device__ __forceinline__ uint32_t vset(const uint32_t *m, int w, int h, int x, int y) {
    return (x <= 0 || x > w || y <= 0 || y > h) ? 0u : (uint32_t)bit_at(m, (y - 1) * w + (x - 1));
}
__device__ __forceinline__ int ms_value(const uint32_t *m, int w, int h, int x, int y) {
    return (int)(vset(m, w, h, x, y) | vset(m, w, h, x + 1, y) << 1 | vset(m, w, h, x, y + 1) << 2 |
                 vset(m, w, h, x + 1, y + 1) << 3);
}

// pDistance (physics_math.cpp:1814-1843) in f32, each operation rounded on
// its own, as the reference's compiled code rounds it.
__device__ float p_distance(float x, float y, float x1, float y1, float x2, float y2) {
#pragma clang fp contract(off)
    const float A = x - x1, B = y - y1, C = x2 - x1, D = y2 - y1;
    const float dot = A * C + B * D;
    const float len_sq = C * C + D * D;
    float param = -1.0f;
    if (len_sq != 0.0f) param = dot / len_sq;
    float xx, yy;
    if (param < 0.0f) {
        xx = x1;
        yy = y1;
    } else if (param > 1.0f) {
        xx = x2;
        yy = y2;
    } else {
        xx = x1 + param * C;
        yy = y1 + param * D;
    }
    const float dx = x - xx, dy = y - yy;
    return sqrtf(dx * dx + dy * dy);
}

__device__ __forceinline__ float vx(uint32_t v) { return (float)(v & 0xFFFFu); }
__device__ __forceinline__ float vy(uint32_t v) { return (float)(v >> 16); }

// Directions of the walk: 0 north (y decreases), 1 east, 2 south, 3 west.
// The next one at a vertex of value v (1 .. 14) after direction prev (4: none).
__device__ __forceinline__ uint32_t walk_dir(uint32_t v, uint32_t prev) {
    //                        14 13 12 11 10  9  8  7  6  5  4  3  2  1 (2 bits each)
    constexpr uint32_t DIRS = 3u << 28 | 0u << 26 | 3u << 24 | 2u << 22 | 2u << 20 | 2u << 18 | 2u << 16 | 1u << 14 |
                              1u << 12 | 0u << 10 | 3u << 8 | 1u << 6 | 1u << 4 | 0u << 2;
    uint32_t d = (DIRS >> (2 * v)) & 3u;
    if (v == 6 && prev == 0) d = 3;
    if (v == 9 && prev == 1) d = 0;
    return d;
}

// Orders one wave's LDS and scratch accesses across its lanes (the workgroup
// scope waits for outstanding stores).
__device__ __forceinline__ void wave_sync() {
    __threadfence_block();
    __builtin_amdgcn_wave_barrier();
}

__device__ __forceinline__ uint32_t wave_prefix(uint32_t v, int lane, uint32_t &total) {  // exclusive
    uint32_t incl = v;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
        const uint32_t u = (uint32_t)__shfl_up((int)incl, off, 64);
        if (lane >= off) incl += u;
    }
    total = (uint32_t)__builtin_amdgcn_readlane((int)incl, 63);
    return incl - v;
}

struct MeshLds {
    uint32_t mask[MWORDS], cand[MWORDS], seen[MWORDS];
    uint8_t value[VCAP];                 // vertex values (small regions), LIVE on the batch's candidates
    uint8_t rank[MBITS];                 // place in the batch of a candidate of it
    uint32_t batch[64];                  // its candidates, in row order
    uint16_t run[2][RUNS * 64];          // run ends (x | y << 8) of the lanes' walks, this batch's and the last one's
    uint16_t start[2][64];               // their start vertices
    uint8_t nrun[2][64];                 // their runs, 0 for walks not kept
    uint16_t sect[(RUNS + 1) * 64];      // RDP sections (i | j << 8) of the simplifying lanes
    uint32_t keep[MAXV / 32 + 1];        // the whole wave's walk: kept runs, run ends, RDP sections
    uint32_t lmesh[LCAP], lstack[LCAP];
    uint32_t nloops, nverts;             // of the region so far
    int big, more;                       // a walk for the whole wave follows; the region is not done
};
static_assert(sizeof(MeshLds) <= 80 * 1024, "two workgroups per compute unit");

// The loop's place in the pools, and its record.  One lane per loop; all lanes
// of the wave call it.
__device__ __forceinline__ bool emit_slot(MeshLds &S, const MeshOut &out, int lane, bool emit, uint32_t ns,
                                          uint32_t start, bool hole, uint32_t region, uint32_t &vslot) {
    const uint64_t m = __ballot(emit);
    if (!m) return false;
    uint32_t nv;
    const uint32_t vo = wave_prefix(emit ? ns : 0u, lane, nv);
    const uint32_t lo = __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u));
    const uint32_t nl = (uint32_t)__popcll(m);
    uint32_t lbase = 0, vbase = 0;
    if (lane == 0) {
        lbase = atomicAdd(&out.counters[0], nl);
        vbase = atomicAdd(&out.counters[1], nv);
    }
    lbase = (uint32_t)__builtin_amdgcn_readfirstlane((int)lbase);
    vbase = (uint32_t)__builtin_amdgcn_readfirstlane((int)vbase);
    const uint32_t l0 = S.nloops, v0 = S.nverts;
    const bool fits = (uint64_t)lbase + nl <= out.loop_cap && (uint64_t)vbase + nv <= out.vert_cap;
    if (!fits && lane == 0) atomicOr(&out.counters[2], 1u);
    if (fits && emit) {
        fsg_mesh_loop L;
        L.first = vbase + vo;
        L.count = ns;
        L.hole = hole ? 1 : 0;
        L.start_x = (int)(start & 0xFFFFu);
        L.start_y = (int)(start >> 16);
        L.region = region;
        out.loops[lbase + lo] = L;
        out.seq[lbase + lo] = l0 + lo;
        out.voff[lbase + lo] = v0 + vo;
    }
    wave_sync();  // every lane has read the region's counts
    if (lane == 0) {
        S.nloops = l0 + nl;
        S.nverts = v0 + nv;
    }
    wave_sync();
    vslot = vbase + vo;
    return fits;
}

// A batch of walks, one per lane of the walking wave.
struct Batch {
    int nb, pos, look;       // its candidates, the next one to judge, where the next batch starts (wave-uniform)
    uint64_t wholes;         // walks that closed
    uint64_t cover;          // this lane's: candidates of the batch its walk marks
    uint32_t p, p0, prev;    // its vertex (x | y << 8), its start, its last direction
    int nr;                  // its runs so far
};

// The next 64 unmarked candidates from B.look on, and each lane's walk.
// Regions of more than 255 cells a side leave the walking to walk_whole.
__device__ void walk_batch(MeshLds &S, int w, int h, bool small, int buf, Batch &B) {
    const int lane = threadIdx.x & 63, size = w * h, nwords = (size + 31) >> 5, most = small ? 64 : 1;
    int nb = 0;
    for (int w0 = B.look >> 5; w0 < nwords && nb < most; w0 += 64) {
        const int wi = w0 + lane;
        uint32_t bits = wi < nwords ? S.cand[wi] & ~S.seen[wi] : 0u;
        if (wi == (B.look >> 5)) bits &= ~0u << (B.look & 31);
        uint32_t total;
        int r = nb + (int)wave_prefix((uint32_t)__popc(bits), lane, total);
        while (bits && r < most) {
            const int i = (wi << 5) + __builtin_ctz(bits);
            bits &= bits - 1;
            S.batch[r] = (uint32_t)i;
            S.rank[i] = (uint8_t)r++;
        }
        nb = min(most, nb + (int)total);
    }
    wave_sync();
    B.nb = nb;
    B.pos = 0;
    B.wholes = 0;
    B.cover = 0;
    B.nr = 0;
    B.prev = 4;
    B.p = B.p0 = 0;
    if (nb == 0) return;
    B.look = (int)S.batch[nb - 1] + 1;
    if (!small) return;
    const uint32_t pitch = (uint32_t)w + 1;
    const int i0 = (int)S.batch[min(lane, nb - 1)];
    const uint32_t y0 = (uint32_t)(i0 / w), x0 = (uint32_t)(i0 - (int)y0 * w);
    // the vertices whose cell (clamped to the region) is this lane's candidate
    auto flag = [&](uint32_t bit) {
        if (lane >= nb) return;
        for (uint32_t y = y0; y <= (y0 + 1 == (uint32_t)h ? y0 + 1 : y0); y++)
            for (uint32_t x = x0; x <= (x0 + 1 == (uint32_t)w ? x0 + 1 : x0); x++)
                S.value[y * pitch + x] = (uint8_t)((S.value[y * pitch + x] & 15u) | bit);
    };
    flag(LIVE);
    wave_sync();
    const uint32_t p0 = x0 | (y0 << 8);
    uint32_t p = p0, prev = 4;
    int nr = 0;
    uint64_t cover = 0;
    bool active = lane < nb, whole = false;
    const int limit = 4 * (w + 1) * (h + 1);
    for (int step = 0; step <= limit && __builtin_amdgcn_ballot_w64(active); step++) {
        if (!active) continue;
        const uint32_t x = p & 255u, y = p >> 8, v = S.value[__umul24(y, pitch) + x], c = v & 15u;
        if (v & LIVE) {
            const uint32_t r = S.rank[min((int)x, w - 1) + min((int)y, h - 1) * w];
            cover |= 1ull << r;
            // an earlier candidate's own vertex, which only its loop passes
            if ((int)r < lane && c != 6 && c != 9 && x < (uint32_t)w && y < (uint32_t)h) active = false;
        }
        const uint32_t d = walk_dir(c, prev);
        const bool turn = d != prev && prev != 4;
        // no perimeter, or no room for this run and the one that closes the loop
        if (c - 1u > 13u || (turn && nr + 1 >= RUNS)) active = false;
        if (!active) continue;  // the walk stands before this step
        if (turn) S.run[buf][nr++ * 64 + lane] = (uint16_t)p;
        const uint32_t one = (d & 1u) ? 1u : 256u;
        p = ((d + 1) & 2u) ? p + one : p - one;
        prev = d;
        whole = p == p0;
        active = !whole;
    }
    if (whole) S.run[buf][nr++ * 64 + lane] = (uint16_t)p0;
    flag(0u);
    B.wholes = __builtin_amdgcn_ballot_w64(whole);
    B.cover = cover;
    B.p = p;
    B.p0 = p0;
    B.prev = prev;
    B.nr = nr;
    wave_sync();
}

// edgeSeen along the runs of the walks with a run count in nrun[buf], a walk
// per lane, every step-th run from k0 on.
__device__ void mark_runs(MeshLds &S, int w, int h, int buf, int k0, int step) {
    const int lane = threadIdx.x & 63, nr = S.nrun[buf][lane];
    for (int k = k0; k < nr; k += step) {
        const uint32_t b = k ? S.run[buf][(k - 1) * 64 + lane] : S.start[buf][lane], e = S.run[buf][k * 64 + lane];
        int sx = (int)(b & 255u), sy = (int)(b >> 8);
        const int ex = (int)(e & 255u), ey = (int)(e >> 8);
        const int ux = (ex > sx) - (ex < sx), uy = (ey > sy) - (ey < sy);
        while (sx != ex || sy != ey) {
            const int ind = min(sx, w - 1) + min(sy, h - 1) * w;
            atomicOr(&S.seen[ind >> 5], 1u << (ind & 31));
            sx += ux;
            sy += uy;
        }
    }
}

// Judges the batch from B.pos on, in row order: the walks the reference makes
// get their run counts (their marks follow, by all waves); stops behind a
// candidate whose walk the whole wave has to finish (S.big).
__device__ void judge_batch(MeshLds &S, int buf, Batch &B) {
    const int lane = threadIdx.x & 63;
    // candidates marked meanwhile by a walk of the whole wave
    const int i0 = B.nb ? (int)S.batch[min(lane, B.nb - 1)] : 0;
    uint64_t kept = 0;
    uint64_t open = __builtin_amdgcn_ballot_w64(lane >= B.pos && lane < B.nb && !bit_at(S.seen, i0));
    int big = -1;
    B.pos = B.nb;
    while (open) {
        const int i = __builtin_ctzll(open);
        if (!((B.wholes >> i) & 1u)) {
            big = i;
            B.pos = i + 1;
            break;
        }
        kept |= 1ull << i;
        open &= ~(1ull << i);
        open &= ~((uint64_t)(uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)B.cover, i) |
                  (uint64_t)(uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(B.cover >> 32), i) << 32);
    }
    S.start[buf][lane] = (uint16_t)B.p0;
    S.nrun[buf][lane] = ((kept >> lane) & 1u) ? (uint8_t)B.nr : (uint8_t)0;
    if (lane == 0) {
        S.big = big;
        S.more = B.nb > 0;
    }
    wave_sync();
}

// The kept walks of a batch, a loop per lane: simplified, oriented, emitted.
__device__ void simplify_batch(MeshLds &S, const MeshOut &out, uint32_t region, int buf) {
    const int lane = threadIdx.x & 63;
    const int nr = S.nrun[buf][lane];
    if (!__builtin_amdgcn_ballot_w64(nr != 0)) return;
    const uint16_t *pt = &S.run[buf][lane];
    auto px = [](uint32_t v) { return (float)(v & 255u); };
    auto py = [](uint32_t v) { return (float)(v >> 8); };
    uint64_t keep = nr ? ~0ull >> (64 - nr) : 0ull;
    int sp = 0;
    if (nr > 2) S.sect[(sp++) * 64 + lane] = (uint16_t)((nr - 1) << 8);
    while (sp > 0) {
        const uint32_t e = S.sect[(--sp) * 64 + lane];
        const int i = (int)(e & 0xFFu), j = (int)(e >> 8);
        if (i + 1 == j) continue;
        const uint32_t vi = pt[i * 64], vj = pt[j * 64];
        float best = -1.0f;
        int bk = i;
        for (int k = i + 1; k < j; k++) {
            const uint32_t vk = pt[k * 64];
            const float d = p_distance(px(vk), py(vk), px(vi), py(vi), px(vj), py(vj));
            if (d > best) {  // the first largest distance
                best = d;
                bk = k;
            }
        }
        if (best <= 1.0f) {
            keep &= ~((~0ull >> (64 - j)) & (~0ull << (i + 1)));  // runs i + 1 .. j - 1
        } else {
            S.sect[(sp++) * 64 + lane] = (uint16_t)((uint32_t)bk | ((uint32_t)j << 8));
            S.sect[(sp++) * 64 + lane] = (uint16_t)((uint32_t)i | ((uint32_t)bk << 8));
        }
    }
    const uint32_t ns = (uint32_t)__popcll(keep);
    const bool emit = ns >= 3;
    // orientation of the reversed list (GetOrientation)
    int area = 0;  // at most 2 * 64 * 255^2
    if (emit) {
        const int last = 63 - __builtin_clzll(keep);
        uint32_t prev = pt[last * 64];
        const uint32_t lastv = prev;
        auto cross = [](uint32_t a, uint32_t b) {
            return (int)(a & 255u) * (int)(b >> 8) - (int)(a >> 8) * (int)(b & 255u);
        };
        for (uint64_t m = keep & ~(1ull << last); m;) {
            const int k = 63 - __builtin_clzll(m);
            m &= ~(1ull << k);
            const uint32_t v = pt[k * 64];
            area += cross(prev, v);
            prev = v;
        }
        area += cross(prev, lastv);
    }
    const uint32_t st = S.start[buf][lane];
    uint32_t vslot;
    if (emit_slot(S, out, lane, emit, ns, (st & 255u) | ((st >> 8) << 16), area < 0, region, vslot) && emit)
        for (uint64_t m = keep; m; m &= m - 1) {
            const uint32_t v = pt[__builtin_ctzll(m) * 64];
            out.verts[vslot++] = (v & 255u) | ((v >> 8) << 16);
        }
}

// Finishes the walk of lane `who` of the batch by the whole wave, in lockstep
// with wave-uniform values; its runs go to LDS up to LCAP, and to the
// workgroup's scratch.
__device__ void walk_whole(MeshLds &S, const MeshOut &out, uint32_t region, int w, int h, bool small, int buf,
                           const Batch &B, int who, uint32_t *gmesh, uint32_t *gstack) {
    const int lane = threadIdx.x & 63;
    const int i0 = (int)S.batch[who], x0 = i0 % w, y0 = i0 / w;
    int x = x0, y = y0, nr = 0, sx = x0, sy = y0;  // vertex, runs so far, start vertex of the open run
    uint32_t prev = 4;
    if (small) {
        // the lane's runs, then its open run
        nr = __builtin_amdgcn_readlane(B.nr, who);
        prev = (uint32_t)__builtin_amdgcn_readlane((int)B.prev, who);
        const uint32_t p = (uint32_t)__builtin_amdgcn_readlane((int)B.p, who);
        x = (int)(p & 255u);
        y = (int)(p >> 8);
        if (lane < nr) {
            const uint32_t b = lane ? S.run[buf][(lane - 1) * 64 + who] : S.start[buf][who];
            const uint32_t e = S.run[buf][lane * 64 + who];
            S.lmesh[lane] = gmesh[lane] = (e & 255u) | ((e >> 8) << 16);
            int bx = (int)(b & 255u), by = (int)(b >> 8);
            const int ex = (int)(e & 255u), ey = (int)(e >> 8);
            const int ux = (ex > bx) - (ex < bx), uy = (ey > by) - (ey < by);
            for (; bx != ex || by != ey; bx += ux, by += uy) {
                const int ind = min(bx, w - 1) + min(by, h - 1) * w;
                atomicOr(&S.seen[ind >> 5], 1u << (ind & 31));
            }
        }
        wave_sync();
        if (nr > 0) {
            const uint32_t e = S.lmesh[nr - 1];
            sx = (int)(e & 0xFFFFu);
            sy = (int)(e >> 16);
        }
    }
    bool ok = true;
    const int limit = 4 * (w + 1) * (h + 1);
    auto close_run = [&]() {  // the open run ends at (x, y)
        const int len = abs(x - sx) + abs(y - sy), ux = (x > sx) - (x < sx), uy = (y > sy) - (y < sy);
        for (int k = lane; k < len; k += 64) {
            const int ind = min(sx + k * ux, w - 1) + min(sy + k * uy, h - 1) * w;
            atomicOr(&S.seen[ind >> 5], 1u << (ind & 31));
        }
        sx = x;
        sy = y;
        if (lane == 0) {
            const uint32_t v = (uint32_t)x | ((uint32_t)y << 16);
            if (nr < LCAP) S.lmesh[nr] = v;
            if (nr < MAXV) gmesh[nr] = v;
        }
        nr++;
    };
    for (int step = 0;; step++) {
        const uint32_t v = small ? S.value[y * (w + 1) + x] & 15u : (uint32_t)ms_value(S.mask, w, h, x, y);
        if (step > limit || v == 0 || v == 15) {
            ok = false;
            break;
        }
        const uint32_t d = walk_dir(v, prev);
        if (prev != 4 && d != prev) close_run();
        prev = d;
        if (d & 1u) x += d == 1 ? 1 : -1;
        else y += d == 2 ? 1 : -1;
        if (x == x0 && y == y0) break;
    }
    if (ok) close_run();
    wave_sync();  // edgeSeen and the runs written
    if (!ok || nr > MAXV) {
        if (lane == 0) atomicAdd(&out.counters[3], 1u);
        return;
    }
    uint32_t *mesh = nr <= LCAP ? S.lmesh : gmesh;
    uint32_t *stack = nr <= LCAP ? S.lstack : gstack;
    // Ramer-Douglas-Peucker, tolerance 1, over mesh[0 .. nr).  Sections of more
    // than SECT runs one at a time, the lanes sharing the search; the others
    // are listed from the array's end (sections are disjoint, so all of them
    // fit in nr entries) and then taken by a lane each.
    for (int k = lane; k < (nr + 31) / 32; k += 64) S.keep[k] = ~0u;
    wave_sync();
    const int room = nr <= LCAP ? LCAP : MAXV;
    int sp = 0, ns_list = 0;
    auto push = [&](int i, int j) {
        if (j - i < 2) return;
        const uint32_t e = (uint32_t)i | ((uint32_t)j << 16);
        if (j - i > SECT) {
            if (lane == 0) stack[sp] = e;
            sp++;
        } else {
            ns_list++;
            if (lane == 0) stack[room - ns_list] = e;
        }
    };
    if (nr > 2) push(0, nr - 1);
    wave_sync();
    while (sp > 0) {
        const uint32_t e = (uint32_t)__builtin_amdgcn_readfirstlane((int)stack[sp - 1]);
        wave_sync();
        sp--;
        const int i = (int)(e & 0xFFFFu), j = (int)(e >> 16);
        const uint32_t vi = mesh[i], vj = mesh[j];
        float best = -1.0f;
        int bk = i;
        for (int k = i + 1 + lane; k < j; k += 64) {
            const uint32_t vk = mesh[k];
            const float d = p_distance(vx(vk), vy(vk), vx(vi), vy(vi), vx(vj), vy(vj));
            if (d > best) {
                best = d;
                bk = k;
            }
        }
        // the first largest distance, as the reference's strict > scan finds it
        for (int off = 32; off > 0; off >>= 1) {
            const float ob = __shfl_xor(best, off, 64);
            const int ok2 = __shfl_xor(bk, off, 64);
            if (ob > best || (ob == best && ok2 < bk)) {
                best = ob;
                bk = ok2;
            }
        }
        if (best <= 1.0f) {
            for (int k = i + 1 + lane; k < j; k += 64) atomicAnd(&S.keep[k >> 5], ~(1u << (k & 31)));
        } else {
            const int m = __builtin_amdgcn_readfirstlane(bk);
            push(m, j);
            push(i, m);
        }
        wave_sync();
    }
    for (int l = lane; l < ns_list; l += 64) {
        const uint32_t e0 = stack[room - 1 - l];
        const int base = (int)(e0 & 0xFFFFu);
        uint16_t *st = &S.sect[lane];  // i | j << 8 from base
        int p = 0;
        st[(p++) * 64] = (uint16_t)(((e0 >> 16) - (uint32_t)base) << 8);
        while (p > 0) {
            const uint32_t e = st[(--p) * 64];
            const int i = base + (int)(e & 0xFFu), j = base + (int)(e >> 8);
            if (i + 1 == j) continue;
            const uint32_t vi = mesh[i], vj = mesh[j];
            float best = -1.0f;
            int bk = i;
            for (int k = i + 1; k < j; k++) {
                const uint32_t vk = mesh[k];
                const float d = p_distance(vx(vk), vy(vk), vx(vi), vy(vi), vx(vj), vy(vj));
                if (d > best) {
                    best = d;
                    bk = k;
                }
            }
            if (best <= 1.0f) {
                for (int k = i + 1; k < j; k++) atomicAnd(&S.keep[k >> 5], ~(1u << (k & 31)));
            } else {
                const uint32_t m = (uint32_t)(bk - base);
                st[(p++) * 64] = (uint16_t)(m | (e & 0xFF00u));
                st[(p++) * 64] = (uint16_t)((e & 0xFFu) | (m << 8));
            }
        }
    }
    wave_sync();
    // kept vertices, compacted to the front of mesh[], in order, 64 at a time
    // (every lane reads before any writes, and writes land at or before the
    // positions read)
    int ns = 0;
    for (int k0 = 0; k0 < nr; k0 += 64) {
        const int k = k0 + lane;
        const bool kp = k < nr && bit_at(S.keep, k);
        const uint32_t v = kp ? mesh[k] : 0u;
        const uint64_t b = __ballot(kp);
        wave_sync();
        if (kp) mesh[ns + (int)__builtin_amdgcn_mbcnt_hi((uint32_t)(b >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)b, 0u))] = v;
        ns += __popcll(b);
        wave_sync();
    }
    if (ns < 3) return;
    // orientation of the reversed list (GetOrientation)
    long long area = 0;
    for (int a = lane; a < ns; a += 64) {
        const int p = ns - 1 - a, q = (a + 1 == ns) ? ns - 1 : ns - 2 - a;
        const uint32_t vp = mesh[p], vq = mesh[q];
        area += (long long)(vp & 0xFFFFu) * (long long)(vq >> 16) - (long long)(vp >> 16) * (long long)(vq & 0xFFFFu);
    }
    for (int off = 32; off > 0; off >>= 1) area += __shfl_xor(area, off, 64);
    uint32_t vslot = 0;
    const bool fits = emit_slot(S, out, lane, lane == 0, (uint32_t)ns, (uint32_t)x0 | ((uint32_t)y0 << 16), area < 0,
                                region, vslot);
    vslot = (uint32_t)__builtin_amdgcn_readfirstlane((int)vslot);
    if (fits)
        for (int k = lane; k < ns; k += 64) out.verts[vslot + k] = mesh[k];
}

__global__ __launch_bounds__(MT) void k_mesh(MeshSrc src, const MeshRegionDev *regs, int nreg, MeshOut out) {
    __shared__ MeshLds S;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    uint32_t *gmesh = out.scratch + (size_t)blockIdx.x * 2 * MAXV;
    uint32_t *gstack = gmesh + MAXV;
    for (int ri = blockIdx.x; ri < nreg; ri += gridDim.x) {
        const MeshRegionDev R = regs[ri];
        const int w = R.w, h = R.h, size = w * h;
        const bool small = w <= 255 && h <= 255;
        // the mask, 64 cells per ballot, four loads of a wave in flight
        constexpr int U = 4;
        for (int b0 = wave * 64; b0 < size; b0 += MT * U) {
            uint32_t m[U];
#pragma unroll
            for (int u = 0; u < U; u++) {
                const int i = b0 + u * MT + lane;
                m[u] = 32;
                if (i < size) {
                    const int y = i / w, x = i - y * w;
                    m[u] = (uint32_t)src.cells[R.off + (int64_t)y * R.pitch + x] & 15u;
                }
            }
#pragma unroll
            for (int u = 0; u < U; u++) {
                const int i0 = b0 + u * MT;
                const uint64_t b = __ballot(m[u] < 32 && ((src.setmask >> (m[u] & 31u)) & 1u));
                if (i0 >= size) continue;
                if (lane == 0) S.mask[i0 >> 5] = (uint32_t)b;
                if (lane == 1 && (i0 >> 5) + 1 < MWORDS) S.mask[(i0 >> 5) + 1] = (uint32_t)(b >> 32);
            }
        }
        if (tid == 0) S.nloops = S.nverts = 0;
        if (tid < 128) S.nrun[tid >> 6][tid & 63] = 0;  // (the first batch has no predecessor)
        __syncthreads();
        // vertex values (last column and row included)
        if (small)
            for (int i = tid; i < (w + 1) * (h + 1); i += MT) {
                const int y = i / (w + 1), x = i - y * (w + 1);
                S.value[i] = (uint8_t)ms_value(S.mask, w, h, x, y);
            }
        // edge candidates (world.cpp:774-789) whose vertex value is neither
        // 0 nor 15 (world.cpp:826-831); edgeSeen cleared
        for (int i0 = wave * 64; i0 < size; i0 += MT) {
            const int i = i0 + lane;
            bool c = false;
            if (i < size && bit_at(S.mask, i)) {
                const int y = i / w, x = i - y * w;
                int nb = 0;
                if (x + 1 < w) nb += bit_at(S.mask, i + 1);
                if (y + 1 < h) nb += bit_at(S.mask, i + w);
                if (y + 1 < h && x + 1 < w) nb += bit_at(S.mask, i + w + 1);
                const int v = ms_value(S.mask, w, h, x, y);
                c = nb != 3 && v != 0 && v != 15;
            }
            const uint64_t b = __ballot(c);
            if (lane == 0) {
                S.cand[i0 >> 5] = (uint32_t)b;
                S.seen[i0 >> 5] = 0u;
            }
            if (lane == 1 && (i0 >> 5) + 1 < MWORDS) {
                S.cand[(i0 >> 5) + 1] = (uint32_t)(b >> 32);
                S.seen[(i0 >> 5) + 1] = 0u;
            }
        }
        __syncthreads();
        // batches: wave 0 walks and judges one while wave 1 simplifies the one
        // before; a walk the whole wave finishes goes out between the loops
        // before it and the rest of its batch (loops go out in trace order)
        Batch B;
        B.nb = B.pos = B.look = 0;
        for (int buf = 0;;) {
            if (wave == 0) {
                if (B.pos >= B.nb) walk_batch(S, w, h, small, buf, B);
                judge_batch(S, buf, B);
            } else if (wave == 1) {
                simplify_batch(S, out, R.region, buf ^ 1);
                S.nrun[buf ^ 1][lane] = 0;
            }
            __syncthreads();
            const bool more = S.more != 0;
            const int big = __builtin_amdgcn_readfirstlane(S.big);
            mark_runs(S, w, h, buf, wave, MT / 64);
            __syncthreads();
            if (!more) break;
            if (big >= 0) {
                if (wave == 1) {
                    simplify_batch(S, out, R.region, buf);
                    S.nrun[buf][lane] = 0;
                }
                __syncthreads();
                if (wave == 0) walk_whole(S, out, R.region, w, h, small, buf, B, big, gmesh, gstack);
                __syncthreads();
            }
            // the rest of a batch stays in its buffer; behind a batch's end the other one is next
            if (big < 0) buf ^= 1;
        }
        if (tid == 0) {
            out.regcnt[R.region] = S.nloops;
            out.regvert[R.region] = S.nverts;
        }
        __syncthreads();
    }
}

// ---- ordering on the device: regions in the caller's order, loops in trace
// order within each ---------------------------------------------------------
// Exclusive scans of the regions' loop and vertex counts, one workgroup.
__global__ __launch_bounds__(1024) void k_mesh_bases(const uint32_t *regcnt, const uint32_t *regvert, uint32_t n,
                                                     uint32_t *regbase, uint32_t *regvbase) {
    __shared__ uint32_t wl[16], wv[16];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    uint32_t cl = 0, cv = 0;  // carried
    for (uint32_t b0 = 0; b0 < n; b0 += 1024) {
        const uint32_t i = b0 + threadIdx.x;
        uint32_t tl, tv;
        const uint32_t el = wave_prefix(i < n ? regcnt[i] : 0u, lane, tl);
        const uint32_t ev = wave_prefix(i < n ? regvert[i] : 0u, lane, tv);
        if (lane == 0) {
            wl[wave] = tl;
            wv[wave] = tv;
        }
        __syncthreads();
        uint32_t bl = cl, bv = cv;
        for (int k = 0; k < 16; k++) {
            if (k < wave) {
                bl += wl[k];
                bv += wv[k];
            }
            cl += wl[k];
            cv += wv[k];
        }
        if (i < n) {
            regbase[i] = bl + el;
            regvbase[i] = bv + ev;
        }
        __syncthreads();
    }
}

// Each pooled loop at its place, with its vertices as float pairs: eight
// lanes per loop.
__global__ __launch_bounds__(256) void k_mesh_emit(MeshOut o, const uint32_t *regbase, const uint32_t *regvbase,
                                                   fsg_mesh_loop *oloops, float2 *overts) {
    if (o.counters[2] | o.counters[3]) return;  // the pools were too small, or a walk failed
    const uint32_t nl = o.counters[0], sub = threadIdx.x & 7u;
    for (uint32_t l = (blockIdx.x * 256u + threadIdx.x) >> 3; l < nl; l += gridDim.x * 32u) {
        fsg_mesh_loop L = o.loops[l];
        const uint32_t from = L.first;
        L.first = regvbase[L.region] + o.voff[l];
        if (sub == 0) oloops[regbase[L.region] + o.seq[l]] = L;
        for (uint32_t v = sub; v < L.count; v += 8) {
            const uint32_t p = o.verts[from + v];
            overts[L.first + v] = make_float2((float)(p & 0xFFFFu), (float)(p >> 16));
        }
    }
}

using fsg_impl::dev_alloc;
using fsg_impl::dev_free;

int grow_buf(fsg_ctx *c, void **p, size_t *cap, size_t bytes) {
    if (*cap >= bytes) return FSG_OK;
    dev_free(*p);
    *p = nullptr;
    *cap = 0;
    if (dev_alloc(c, p, bytes)) return FSG_ERR_NOMEM;
    *cap = bytes;
    return FSG_OK;
}

// Runs the mesher over regions (already validated) and leaves the ordered
// result in w->mesh_loops / w->mesh_verts.
int run_mesh(fsg_world *w, const MeshSrc &src, std::vector<MeshRegionDev> &regs, fsg_mesh_region *out_regions,
             int nout, uint32_t *nloops, uint32_t *nverts) {
    fsg_ctx *c = w->ctx;
    HIPCHK(hipSetDevice(c->device));
    w->mesh_nloops = 0;
    w->mesh_nverts = 0;
    for (int i = 0; i < nout; i++) {
        out_regions[i].first_loop = 0;
        out_regions[i].nloops = 0;
    }
    const int n = (int)regs.size();
    if (n > 0) {
        const int grid = std::min(n, 1024);
        auto al = [](size_t b) { return (b + 255) & ~(size_t)255; };
        // the region table; then the counters and the regions' loop counts
        // (one copy to the host), their vertex counts, and the scans of both
        const size_t b_regs = al((size_t)n * sizeof(MeshRegionDev)), b_out = 16 + (size_t)nout * 4;
        if (grow_buf(c, &w->d_mesh_regs, &w->mesh_regs_cap, b_regs + b_out + 3 * (size_t)nout * 4) ||
            grow_buf(c, &w->d_mesh_scratch, &w->mesh_scratch_cap, (size_t)grid * 2 * MAXV * 4))
            return FSG_ERR_NOMEM;
        MeshOut o;
        o.counters = reinterpret_cast<unsigned int *>(static_cast<char *>(w->d_mesh_regs) + b_regs);
        o.regcnt = o.counters + 4;
        o.regvert = o.regcnt + nout;
        uint32_t *regbase = o.regvert + nout, *regvbase = regbase + nout;
        if (int rc = fsg_impl::copy_in(c, w->d_mesh_regs, regs.data(), (size_t)n * sizeof(MeshRegionDev))) return rc;
        // pools sized from the last call, grown and the launch repeated on overflow
        uint32_t loop_cap = std::max<uint32_t>(w->mesh_loop_hint, 4096u);
        uint32_t vert_cap = std::max<uint32_t>(w->mesh_vert_hint, 65536u);
        bool done = false;
        std::vector<uint32_t> h(b_out / 4);
        for (int attempt = 0; attempt < 2 && !done; attempt++) {
            // the pool: traced loops, their seq and vertex offsets, vertices;
            // then the ordered loops and vertices
            const size_t b_loops = al((size_t)loop_cap * sizeof(fsg_mesh_loop)), b_l4 = al((size_t)loop_cap * 4);
            const size_t b_v4 = al((size_t)vert_cap * 4);
            const size_t total = 2 * b_loops + 2 * b_l4 + b_v4 + al((size_t)vert_cap * 8);
            if (grow_buf(c, &w->d_mesh_pool, &w->mesh_pool_cap, total)) return FSG_ERR_NOMEM;
            char *pool = static_cast<char *>(w->d_mesh_pool);
            o.loops = reinterpret_cast<fsg_mesh_loop *>(pool);
            pool += b_loops;
            o.seq = reinterpret_cast<uint32_t *>(pool);
            pool += b_l4;
            o.voff = reinterpret_cast<uint32_t *>(pool);
            pool += b_l4;
            o.verts = reinterpret_cast<uint32_t *>(pool);
            pool += b_v4;
            fsg_mesh_loop *oloops = reinterpret_cast<fsg_mesh_loop *>(pool);
            pool += b_loops;
            float2 *overts = reinterpret_cast<float2 *>(pool);
            o.loop_cap = loop_cap;
            o.vert_cap = vert_cap;
            o.scratch = static_cast<uint32_t *>(w->d_mesh_scratch);
            HIPCHK(hipMemsetAsync(o.counters, 0, b_out + (size_t)nout * 4, c->stream));
            k_mesh<<<grid, MT, 0, c->stream>>>(src, static_cast<const MeshRegionDev *>(w->d_mesh_regs), n, o);
            k_mesh_bases<<<1, 1024, 0, c->stream>>>(o.regcnt, o.regvert, (uint32_t)nout, regbase, regvbase);
            k_mesh_emit<<<std::min<uint32_t>((loop_cap + 31) / 32, 2048u), 256, 0, c->stream>>>(o, regbase, regvbase,
                                                                                               oloops, overts);
            HIPCHK(hipGetLastError());
            if (int rc = fsg_impl::copy_out(c, {{h.data(), o.counters, b_out}})) return rc;
            const uint32_t *cnt = h.data(), *rc = cnt + 4;
            if (cnt[3]) return FSG_ERR_DEVICE;  // a walk that did not close: not a perimeter of a finite mask
            if (cnt[2]) {
                loop_cap = std::max(loop_cap, cnt[0] + 1024u);
                vert_cap = std::max(vert_cap, cnt[1] + 65536u);
                continue;
            }
            w->mesh_loop_hint = cnt[0];
            w->mesh_vert_hint = cnt[1];
            uint32_t first = 0;
            for (int r = 0; r < nout; r++) {
                out_regions[r].first_loop = rc[r] ? first : 0;
                out_regions[r].nloops = rc[r];
                first += rc[r];
            }
            w->d_mesh_loops = oloops;
            w->d_mesh_verts = reinterpret_cast<float *>(overts);
            w->mesh_nloops = cnt[0];
            w->mesh_nverts = cnt[1];
            done = true;
        }
        if (!done) return FSG_ERR_NOMEM;  // the second launch had pools of the first one's totals
    }
    if (nloops) *nloops = w->mesh_nloops;
    if (nverts) *nverts = w->mesh_nverts;
    return FSG_OK;
}

uint32_t type_mask(const fsg_config &cfg, bool solid) {
    uint32_t m = 0;
    for (uint32_t i = 0; i < cfg.n_materials; i++) {
        const uint8_t t = cfg.materials[i].type;
        if (solid ? t == FSG_SOLID : t != FSG_AIR) m |= 1u << i;
    }
    if (solid) m |= 1u << fsg::WALL;
    return m;
}

}  // namespace

extern "C" int fsg_world_mesh(fsg_world *w, fsg_mesh_region *regions, int n, uint32_t *nloops, uint32_t *nverts) {
    if (!w || n < 0 || (n && !regions)) return FSG_ERR_INVALID;
    std::vector<MeshRegionDev> regs;
    for (int i = 0; i < n; i++) {
        fsg_mesh_region &R = regions[i];
        if (R.w <= 0 || R.h <= 0 || (int64_t)R.w * R.h > FSG_MESH_MAX_CELLS) return FSG_ERR_INVALID;
    }
    for (int i = 0; i < n; i++) {
        fsg_mesh_region &R = regions[i];
        // the reference meshes a chunk only when it ends before the world's
        // last row and column (world.cpp:734-736)
        if (R.x0 < 0 || R.y0 < 0 || (int64_t)R.x0 + R.w >= w->d.W || (int64_t)R.y0 + R.h >= w->d.H) {
            R.status = FSG_MESH_EDGE;
            continue;
        }
        R.status = FSG_OK;
        regs.push_back(MeshRegionDev{(int64_t)R.y0 * w->d.W + R.x0, w->d.W, R.w, R.h, (uint32_t)i});
    }
    MeshSrc src{w->d.buf[w->d.tick & 1], type_mask(w->cfg, true)};
    return run_mesh(w, src, regs, regions, n, nloops, nverts);
}

extern "C" int fsg_world_mesh_islands(fsg_world *w, const fsg_island *islands, int n, fsg_mesh_region *regions,
                                      uint32_t *nloops, uint32_t *nverts) {
    if (!w || n < 0 || (n && (!islands || !regions))) return FSG_ERR_INVALID;
    std::vector<MeshRegionDev> regs;
    for (int i = 0; i < n; i++) {
        const fsg_island &I = islands[i];
        fsg_mesh_region &R = regions[i];
        R.x0 = 0;
        R.y0 = 0;
        R.w = I.w;
        R.h = I.h;
        // no outline for other statuses, or for an image one pixel wide or
        // high (world.cpp:331, 365)
        if (I.status != FSG_ISLAND_BODY || I.w <= 1 || I.h <= 1) {
            R.status = FSG_MESH_EDGE;
            continue;
        }
        if ((int64_t)I.w * I.h > FSG_MESH_MAX_CELLS ||
            I.pixel_offset + (uint64_t)I.w * I.h > (uint64_t)w->isl_pix_used)
            return FSG_ERR_INVALID;
        R.status = FSG_OK;
        regs.push_back(MeshRegionDev{(int64_t)I.pixel_offset, I.w, I.w, I.h, (uint32_t)i});
    }
    MeshSrc src{w->d_isl_pix, type_mask(w->cfg, false)};
    return run_mesh(w, src, regs, regions, n, nloops, nverts);
}

extern "C" int fsg_world_mesh_download(fsg_world *w, fsg_mesh_loop *loops, uint32_t loop_cap, float *verts,
                                       uint32_t vert_cap) {
    if (!w) return FSG_ERR_INVALID;
    const size_t nl = w->mesh_nloops, nv = w->mesh_nverts;
    if ((nl && (!loops || loop_cap < nl)) || (nv && (!verts || vert_cap < nv))) return FSG_ERR_INVALID;
    fsg_ctx *c = w->ctx;
    HIPCHK(hipSetDevice(c->device));
    return fsg_impl::copy_out(c, {{loops, w->d_mesh_loops, nl * sizeof(fsg_mesh_loop)},
                                  {verts, w->d_mesh_verts, nv * 2 * sizeof(float)}});
}
