// fsg_particles.hip -- free-fall particles (CellData, game_utils/cells.h:15-36)
// and world::tickCells (world.cpp:2030-2189) on the device.
//
// The reference moves its particles one after another, and a particle that
// lands changes the cells the particles after it move through and search:
// particle i's outcome is a function of the grid and of the landings of the
// particles before it.  The device finds those outcomes as a fixed point.
// Every particle moves in parallel against the grid plus a view of the
// landings the previous round found, in which a landing counts for particle
// i only if an earlier particle made it (a hash of landing cell -> lowest
// index).  A round whose landings equal the previous round's has the
// outcomes the sequential order gives: by induction over the list, each
// particle saw exactly the landings before it.  After any round the particles
// before the first one whose landing changed are already final, so the next
// round moves only the rest; a round with no landing change ends the pass.
// A list whose rounds keep changing (a long chain of landings that depend on
// each other) hands its unfinished part to the batch walk below, which keeps
// the order by construction.
//
// Batch walk: one workgroup walks the list in batches of 256: every lane
// moves its particle against the grid as the earlier batches left it, and
// records the bounding box of every cell it read (its path, the cell it
// started in, the spiral it searched).  A lane whose box holds the landing
// cell of an earlier lane of the batch might have seen something else had it
// run after that lane; the first such lane ends the batch, the lanes before
// it commit, and the next batch starts at it.
#include "fsg_internal.hpp"

#include <algorithm>
#include <cmath>

namespace {

constexpr int PT = 256;  // particles per batch (threads of the one workgroup)
constexpr int NSPIRAL = 1024;

// tickCells' landing spiral (world.cpp:2113-2139), walked in place: from
// (0, 0) heading (0, -1), turning left where x == y, or x < 0 and x == -y,
// or x > 0 and x == 1 - y.  Its 1024 steps stay within [-15, 16]^2.  (Walking
// it costs a few VALU a step; a table read per step is a memory latency in
// the divergent search loop.)
struct Spiral {
    int x = 0, y = 0, dx = 0, dy = -1;
    __device__ __forceinline__ void next() {
        if (x == y || (x < 0 && x == -y) || (x > 0 && x == 1 - y)) {
            const int t = dx;
            dx = -dy;
            dy = t;
        }
        x += dx;
        y += dy;
    }
};

struct PState {
    fsg_particle p;
    int kind;         // 0 keep, 1 drop, 2 land
    int land;         // cell index of a landing
    int bx0, by0, bx1, by1;  // bounding box of the cells read
};

__device__ __forceinline__ void grow_box(PState &s, int x, int y) {
    s.bx0 = min(s.bx0, x);
    s.by0 = min(s.by0, y);
    s.bx1 = max(s.bx1, x);
    s.by1 = max(s.by1, y);
}

__device__ __forceinline__ bool is_air(const uint64_t *cells, uint32_t airmask, int i) {
    return (airmask >> (uint32_t)(cells[i] & 15u)) & 1u;
}

// Landings seen by particle `self`: slots[h].x = landing cell (EMPTY: free slot),
// .y = lowest index of a particle that landed there with a non-air tile.
// slots == nullptr: no landings.
constexpr uint32_t EMPTY = 0xFFFFFFFFu;
struct View {
    const uint2 *slots;
    uint32_t mask, self;
};

__device__ __forceinline__ uint32_t slot_of(uint32_t cell, uint32_t mask) { return fsg::lowbias32(cell) & mask; }

// Whether an earlier particle landed in cell i; q: the slot at i's hash, h.
__device__ __forceinline__ bool taken(const View &v, uint32_t i, uint32_t h, uint2 q) {
    for (;;) {  // the table is at most half full
        if (q.x == EMPTY) return false;
        if (q.x == i) return q.y < v.self;
        h = (h + 1) & v.mask;
        q = v.slots[h];
    }
}

// An air cell of the grid that no earlier particle has filled.
__device__ __forceinline__ bool free_cell(const uint64_t *cells, uint32_t airmask, const View &v, int i) {
    if (!is_air(cells, airmask, i)) return false;
    if (!v.slots) return true;
    const uint32_t h = slot_of((uint32_t)i, v.mask);
    return !taken(v, (uint32_t)i, h, v.slots[h]);
}

// Which 8 x 8 blocks of the grid hold an air cell, found on demand: two bits
// per block in one word (bit 2k: known, bit 2k + 1: air), so one atomicOr
// publishes both.  Cleared at the start of a pass; the grid only loses air
// cells during a pass, so a block once known to hold none never gains one.
struct AirMap {
    uint32_t *bits;  // null: no map
    int wpr;         // words per block row (16 blocks a word)
};

__device__ bool block_has_air(const AirMap &am, const uint64_t *cells, int W, int H, uint32_t airmask, int bx,
                              int by) {
    uint32_t *wd = am.bits + (size_t)by * am.wpr + (bx >> 4);
    const uint32_t sh = 2u * (uint32_t)(bx & 15);
    const uint32_t v = *wd;
    if ((v >> sh) & 1u) return (v >> (sh + 1)) & 1u;
    bool air = false;
    const int x0 = bx * 8, y0 = by * 8, x1 = min(x0 + 8, W), y1 = min(y0 + 8, H);
    if (x1 - x0 == 8 && y1 - y0 == 8 && (W & 1) == 0) {
        // a whole block of an even-width grid: four rounds of eight 16-byte
        // loads issued together (two rows each)
#pragma unroll 1
        for (int r2 = 0; r2 < 4; r2++) {
            uint4 q[8];
#pragma unroll
            for (int k = 0; k < 8; k++)
                q[k] = *reinterpret_cast<const uint4 *>(cells + (size_t)(y0 + 2 * r2 + (k >> 2)) * W + x0 + 2 * (k & 3));
#pragma unroll
            for (int k = 0; k < 8; k++) air |= ((airmask >> (q[k].x & 15u)) | (airmask >> (q[k].z & 15u))) & 1u;
        }
    } else {
        for (int y = y0; y < y1; y++)
            for (int x = x0; x < x1; x++) air |= (airmask >> (uint32_t)(cells[(size_t)y * W + x] & 15u)) & 1u;
    }
    atomicOr(wd, (1u | (air ? 2u : 0u)) << sh);
    return air;
}

// Bit planes of the grid for the rounds (which only read it): one bit per cell
// that holds air, and one per cell that some landing of the view is in, so
// that a step of a path is two loads that stay in the L2 and the view's hash
// is searched only where a landing is.
struct BitMaps {
    const uint32_t *air;     // null: not built
    const uint32_t *landed;  // null: no landings
    int wpr;                 // words per row
};

// free_cell for a cell (x, y) of the grid, from its words of the planes.
__device__ __forceinline__ bool free_word(uint32_t a, uint32_t l, const View &v, int x, int y, int W) {
    if (!((a >> (x & 31)) & 1u)) return false;
    if (!((l >> (x & 31)) & 1u)) return true;
    const uint32_t i = (uint32_t)(x + y * W), h = slot_of(i, v.mask);
    return !taken(v, i, h, v.slots[h]);
}

__device__ __forceinline__ bool free_bit(const BitMaps &bm, const View &v, int x, int y, int W) {
    const size_t w = (size_t)y * bm.wpr + (x >> 5);
    return free_word(bm.air[w], bm.landed ? bm.landed[w] : 0u, v, x, y, W);
}

// Index of offset (x, y) on the spiral: ring r starts right of its lower right
// corner and runs up the right side, left along the top, down the left side
// and right along the bottom.
__device__ __forceinline__ uint32_t spiral_index(int x, int y) {
    const int r = max(abs(x), abs(y));
    const int side = (x == r && y > -r) ? y + r - 1 : y == r ? 3 * r - 1 - x : x == -r ? 5 * r - 1 - y : 7 * r - 1 + x;
    return r ? (uint32_t)((2 * r - 1) * (2 * r - 1) + side) : 0u;
}

// First cell on the spiral among row y's cells `b` (bit k: offset k - 15), as
// index << 5 | bit; NO_CELL if b is empty.  The row's middle |x| <= |y| is part
// of one ring's top, walked leftwards, or bottom, walked rightwards; the rest
// are rings further out, on whose right side they come before the left.
constexpr uint32_t NO_CELL = 0xFFFFu;
__device__ __forceinline__ uint32_t first_of_row(uint32_t b, int y) {
    if (!b) return NO_CELL;
    const int a = abs(y);
    const uint32_t hi = (a >= 16 ? 0u : ~1u << (15 + a)), lo = a >= 15 ? 0u : (1u << (15 - a)) - 1u;
    const uint32_t mid = b & ~(hi | lo);
    int k;
    if (mid) {
        k = y > 0 ? 31 - __builtin_clz(mid) : __builtin_ctz(mid);
    } else {
        const int r = (b & hi) ? __builtin_ctz(b & hi) : 99, l = (b & lo) ? 31 - __builtin_clz(b & lo) : -99;
        k = r - 15 <= 15 - l ? r : l;
    }
    return spiral_index(k - 15, y) << 5 | (uint32_t)k;
}

// The landing search from the planes.  The 32 x 32 offsets of the spiral are a
// window of the air plane: its rows go into LDS with each row's first cell on
// the spiral beside them (`rows`, `firsts`: the lane's columns), so the next
// candidate is a minimum over 32 numbers instead of a walk of up to 1024
// steps; one taken by an earlier landing is removed from its row.  Walking the
// window's bits in spiral order instead: 65 us a round for 40 000 particles on
// 4096^2, with this 24; reading the grid's cells in spiral order: 233.
// (int)(x + offset) is (int)x + offset for all offsets unless a sum rounds up
// to the next integer, which the largest sum shows; sums in (-1, 0) give cell 0
// again, right before or after its own offset or later.  Returns the landing
// cell or -1, and grows the box over what it read.
__device__ __forceinline__ int search_bits(PState &s, float cx0, float cy0, int W, int H, const View &view,
                                           const BitMaps &bm, uint32_t *rows, uint16_t *firsts) {
    const int mx = (int)cx0, my = (int)cy0;
    int land = -1, reach = 16;
    if ((int)(cx0 + 16.0f) == mx + 16 && (int)(cy0 + 16.0f) == my + 16 && max(mx, my) < (1 << 23) - 16) {
        const int ox = mx - 15, w0 = max(ox, 0) >> 5, sh = max(ox, 0) & 31, up = max(-ox, 0);
        const bool two = w0 + 1 < bm.wpr;
        uint32_t best = ~0u;
        for (int r0 = 0; r0 < 32; r0 += 8) {
            uint32_t lo[8], hi[8];
#pragma unroll
            for (int u = 0; u < 8; u++) {
                const int y = my - 15 + r0 + u;
                const bool in = y >= 0 && y < H;
                const uint32_t *q = bm.air + (size_t)max(y, 0) * bm.wpr + w0;
                lo[u] = in ? q[0] : 0u;
                hi[u] = (in && two) ? q[1] : 0u;
            }
#pragma unroll
            for (int u = 0; u < 8; u++) {
                const uint32_t b = (uint32_t)((((uint64_t)hi[u] << 32) | lo[u]) >> sh) << up;
                const uint32_t f = first_of_row(b, r0 + u - 15);
                rows[(r0 + u) * 256] = b;
                firsts[(r0 + u) * 256] = (uint16_t)f;
                best = min(best, f << 5 | (uint32_t)(r0 + u));
            }
        }
        // one candidate, then four at a time: their slots are loaded together
        for (int some = 1; (best >> 5) != NO_CELL && land < 0; some = 4) {
            int at[4];
            uint32_t h[4];
            uint2 q[4];
#pragma unroll
            for (int u = 0; u < 4; u++) {
                at[u] = -1;
                q[u] = make_uint2(EMPTY, 0u);
                if (u >= some || (best >> 5) == NO_CELL) continue;
                const int row = (int)(best & 31u), k = (int)(best >> 5 & 31u);
                at[u] = row << 5 | k;
                if (!view.slots) break;  // every air cell is free
                const uint32_t i = (uint32_t)(mx + k - 15 + (my + row - 15) * W);
                h[u] = slot_of(i, view.mask);
                q[u] = view.slots[h[u]];
                const uint32_t b = rows[row * 256] & ~(1u << k);
                rows[row * 256] = b;
                firsts[row * 256] = (uint16_t)first_of_row(b, row - 15);
                best = ~0u;
#pragma unroll
                for (int r = 0; r < 32; r++) best = min(best, (uint32_t)firsts[r * 256] << 5 | (uint32_t)r);
            }
#pragma unroll
            for (int u = 0; u < 4; u++) {
                if (at[u] < 0 || land >= 0) continue;
                const int x = (at[u] & 31) - 15, y = (at[u] >> 5) - 15;
                const uint32_t i = (uint32_t)(mx + x + (my + y) * W);
                if (view.slots && taken(view, i, h[u], q[u])) continue;
                land = (int)i;
                reach = max(abs(x), abs(y));
            }
        }
    } else {
        Spiral sp;
        for (int k = 0; k < NSPIRAL && land < 0; k++) {
            const int cx = (int)(cx0 + (float)sp.x), cy = (int)(cy0 + (float)sp.y);
            sp.next();
            if (cx < 0 || cy < 0 || cx >= W || cy >= H) continue;  // the reference reads out of range here
            if (free_bit(bm, view, cx, cy, W)) land = cx + cy * W;
        }
    }
    // everything read lies within the ring reached (a cell more for rounding)
    grow_box(s, max(mx - reach - 1, 0), max(my - reach - 1, 0));
    grow_box(s, min(mx + reach + 1, W - 1), min(my + reach + 1, H - 1));
    return land;
}

// One particle's tick against the grid (the reference's loop body).  BITS: the
// cells are read from the planes bm (rows, firsts: the lane's columns of the
// search window in LDS), else from the grid and the on-demand map am.
template <bool BITS>
__device__ void move_particle(PState &s, const uint64_t *cells, int W, int H, uint32_t airmask, int4 zone,
                              const View &view, const AirMap &am, const BitMaps &bm = BitMaps{},
                              uint32_t *rows = nullptr, uint16_t *firsts = nullptr) {
#pragma clang fp contract(off)
    fsg_particle c = s.p;
    s.kind = 0;
    s.land = -1;
    s.bx0 = s.by0 = 1 << 30;
    s.bx1 = s.by1 = -(1 << 30);
    if ((c.flags & FSG_PARTICLE_TEMPORARY) && c.lifetime <= 0) {
        s.kind = 1;
        return;
    }
    if (c.target_force != 0.0f) {
        const float tdx = c.target_x - c.x, tdy = c.target_y - c.y;
        const float nf = sqrtf(tdx * tdx + tdy * tdy);
        c.vx += tdx / nf * c.target_force;
        c.vy += tdy / nf * c.target_force;
        if (nf < 100.0f) {
            c.vx *= 0.95f;
            c.vy *= 0.95f;
        }
    }
    const int lx = (int)c.x, ly = (int)c.y;
    if (c.x < 0.0f || (int)c.x >= W || c.y < 0.0f || (int)c.y >= H) {
        s.kind = 1;
        return;
    }
    if (lx < zone.x || ly < zone.y || lx >= zone.z || ly >= zone.w) {  // outside the tick zone: kept as it is
        s.p = c;
        return;
    }
    c.vx += c.ax;
    c.vy += c.ay;
    const int div = (int)((fabsf(c.vx) + fabsf(c.vy)) + 1.0f);
    const float dvx = c.vx / (float)div, dvy = c.vy / (float)div;
    bool done = false;
    // BITS: the plane's words of the next four steps are loaded together
    constexpr int AHEAD = 4;
    uint32_t wa[AHEAD], wl[AHEAD];
    for (int k = 0; k < div && !done; k++) {
        if (BITS && (k & (AHEAD - 1)) == 0) {
            float qx = c.x, qy = c.y;
#pragma unroll
            for (int u = 0; u < AHEAD; u++) {
                qx += dvx;
                qy += dvy;
                const bool in = !(qx < 0.0f || (int)qx >= W || qy < 0.0f || (int)qy >= H);
                const size_t wd = in ? (size_t)(int)qy * bm.wpr + ((int)qx >> 5) : 0;
                wa[u] = bm.air[wd];
                wl[u] = bm.landed ? bm.landed[wd] : 0u;
            }
        }
        c.x += dvx;
        c.y += dvy;
        if (c.x < 0.0f || (int)c.x >= W || c.y < 0.0f || (int)c.y >= H) {
            s.kind = 1;
            return;
        }
        const int px = (int)c.x, py = (int)c.y;
        if (c.flags & FSG_PARTICLE_PHASE) continue;
        grow_box(s, px, py);
        const int u = k & (AHEAD - 1);
        if (BITS ? free_word(u == 0 ? wa[0] : u == 1 ? wa[1] : u == 2 ? wa[2] : wa[3],
                             u == 0 ? wl[0] : u == 1 ? wl[1] : u == 2 ? wl[2] : wl[3], view, px, py, W)
                 : free_cell(cells, airmask, view, px + py * W)) continue;
        if (c.in_object_state <= 1) c.in_object_state = 2;  // no OBJECT cells on this grid
        done = true;
        if (c.flags & FSG_PARTICLE_TEMPORARY) {
            s.kind = 1;
            return;
        }
        grow_box(s, lx, ly);
        if (!(BITS ? free_bit(bm, view, lx, ly, W) : free_cell(cells, airmask, view, lx + ly * W))) {
            if (BITS) {
                s.land = search_bits(s, c.x, c.y, W, H, view, bm, rows, firsts);
                if (s.land >= 0) {
                    s.kind = 2;
                    return;
                }
                c.vy = -4.0f;
                c.y -= 16.0f;
                continue;
            }
            // SB offsets at a time: their cells are loaded together, then
            // tested in spiral order.  After the first SB, a 5 x 5 mask of the
            // 8 x 8 blocks the spiral can reach says which hold an air cell;
            // offsets in the others are not loaded (no cell there is free),
            // and with no air block the search ends at once.
            constexpr int SB = 16;
            uint32_t m25 = 0;
            int bx0 = 0, by0 = 0;
            bool masked = false;
            Spiral sp;
            for (int k0 = 0; k0 < NSPIRAL; k0 += SB) {
                if (k0 == SB && am.bits) {
                    // the spiral reads cells of [(int)(x - 15), (int)(x + 16)] x
                    // [(int)(y - 15), (int)(y + 16)] (the float sums are monotone in
                    // the offset), at most 5 blocks each way
                    const int xa = max((int)(c.x + -15.0f), 0), xb = min((int)(c.x + 16.0f), W - 1);
                    const int ya = max((int)(c.y + -15.0f), 0), yb = min((int)(c.y + 16.0f), H - 1);
                    bx0 = xa >> 3;
                    by0 = ya >> 3;
                    for (int by = by0; by <= (yb >> 3); by++)
                        for (int bx = bx0; bx <= (xb >> 3); bx++)
                            if (block_has_air(am, cells, W, H, airmask, bx, by)) m25 |= 1u << ((by - by0) * 5 + (bx - bx0));
                    grow_box(s, xa, ya);  // the rest of the search reads within the rectangle
                    grow_box(s, xb, yb);
                    if (!m25) break;
                    masked = true;
                }
                int at[SB];
                uint32_t m[SB];
#pragma unroll
                for (int u = 0; u < SB; u++) {
                    const int cx = (int)(c.x + (float)sp.x);
                    const int cy = (int)(c.y + (float)sp.y);
                    sp.next();
                    bool in = cx >= 0 && cy >= 0 && cx < W && cy < H;  // the reference reads out of range here
                    if (masked && in) in = (m25 >> (((cy >> 3) - by0) * 5 + ((cx >> 3) - bx0))) & 1u;
                    at[u] = in ? cx + cy * W : -1;
                    m[u] = in ? (uint32_t)cells[cx + cy * W] : 0u;
                    if (in && !masked) grow_box(s, cx, cy);
                }
#pragma unroll
                for (int u = 0; u < SB; u++) {
                    if (at[u] < 0 || !((airmask >> (m[u] & 15u)) & 1u)) continue;
                    if (free_cell(cells, airmask, view, at[u])) {
                        s.kind = 2;
                        s.land = at[u];
                        return;
                    }
                }
            }
            c.vy = -4.0f;
            c.y -= 16.0f;
        } else {
            s.kind = 2;
            s.land = lx + ly * W;
            return;
        }
    }
    if (!done && c.lifetime > 0) c.lifetime--;
    s.p = c;
}

struct PArgs {
    fsg_particle *p;       // the list, updated in place
    uint8_t *alive;        // per particle: kept after the pass
    uint32_t start;        // first particle not yet final
    uint32_t n;
    uint64_t *cells;
    int W, H, tiles_x;
    uint32_t airmask;
    int4 zone;             // tick zone [x, z) x [y, w)
    uint32_t *flags;       // chunk flags the next tick reads (null: no skipping)
    unsigned long long *landed;
    uint32_t *airbits;     // the pass's air-block map
    int air_wpr;
};

__global__ __launch_bounds__(PT) void k_particles(PArgs a) {
    __shared__ int land_at[PT];
    __shared__ int first_bad, next;
    const int t = threadIdx.x;
    uint32_t base = a.start;
    unsigned long long nl = 0;
    const View none{nullptr, 0u, 0u};
    const AirMap am{a.airbits, a.air_wpr};
    while (base < a.n) {  // base is the same in every thread
        const uint32_t i = base + (uint32_t)t;
        PState s;
        const bool mine = i < a.n;
        if (mine) {
            s.p = a.p[i];
            move_particle<false>(s, a.cells, a.W, a.H, a.airmask, a.zone, none, am);
        }
        land_at[t] = (mine && s.kind == 2) ? s.land : -1;
        if (t == 0) first_bad = PT;
        __syncthreads();
        // the first lane whose reads cover an earlier lane's landing
        bool bad = false;
        if (mine && s.bx0 <= s.bx1) {
            for (int j = 0; j < t && !bad; j++) {
                const int c = land_at[j];
                if (c < 0) continue;
                const int cy = c / a.W, cx = c - cy * a.W;
                bad = cx >= s.bx0 && cx <= s.bx1 && cy >= s.by0 && cy <= s.by1;
            }
        }
        if (bad) atomicMin(&first_bad, t);
        __syncthreads();
        const int fb = first_bad;
        if (mine && t < fb) {
            if (s.kind == 2) {
                const fsg_cell &tl = s.p.tile;
                a.cells[s.land] = (uint64_t)tl.mat | ((uint64_t)(uint16_t)tl.temp << 16) | ((uint64_t)tl.rgba << 32);
                if (a.flags) {
                    const int cy = s.land / a.W, cx = s.land - cy * a.W;
                    atomicOr(&a.flags[(cy / fsg::TH) * a.tiles_x + cx / fsg::TW], fsg::F_WAKE_ALL);
                }
                nl++;
            }
            a.alive[i] = s.kind == 0 && !(s.p.y > (float)a.H);  // erase_if(y > height), world.cpp:2190
            if (s.kind == 0) a.p[i] = s.p;
        }
        if (t == 0) next = (int)min((uint32_t)fb, a.n - base);
        __syncthreads();
        base += (uint32_t)next;
        __threadfence_block();  // the landings are seen by the next batch's loads
        __syncthreads();
    }
    for (int off = 32; off > 0; off >>= 1) nl += __shfl_xor(nl, off, 64);
    if ((t & 63) == 0 && nl) atomicAdd(a.landed, nl);
}

// ---- fixed-point rounds ------------------------------------------------------
struct PRes {
    fsg_particle p;  // state if kept
    int32_t kind;    // 0 keep, 1 drop, 2 land
    int32_t land;    // landing cell
    int32_t bx0, by0, bx1, by1;  // bounding box of the cells it read
};

__global__ void k_u32_fill(uint32_t *p, uint32_t n, uint32_t v) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = v;
}

// The landings of a round: a hash of landing cell -> lowest index and, where the
// planes are built, the bit plane of its cells.
struct Table {
    uint2 *slots;
    uint32_t *landed;
};

struct PrepArgs {
    const uint64_t *cells;
    int W, H;
    uint32_t airmask;
    uint32_t *bits;  // the air plane (null: not built)
    int wpr;
    uint32_t bit_words, hcap, n, ncnt;
    Table t[2];
    int32_t *vkey;
    uint32_t *cnt;
    unsigned long long *totals;
};

// Start of a pass, one launch: the air plane from the grid (a wave takes 64
// columns of eight rows, so its loads are independent: bound by the read, 23
// us for 4096^2, 5.7 TB/s), empty tables, no landings, counters at zero.
__global__ __launch_bounds__(256) void k_ph_prep(PrepArgs a) {
    const uint32_t i0 = blockIdx.x * 256 + threadIdx.x, step = gridDim.x * 256;
    if (a.bits) {
        constexpr int R = 8;
        const int lane = threadIdx.x & 63;
        const uint32_t nbx = (uint32_t)a.wpr / 2, nby = ((uint32_t)a.H + R - 1) / R;
        for (uint32_t b = blockIdx.x * 4 + (threadIdx.x >> 6); b < nbx * nby; b += gridDim.x * 4) {
            const uint32_t by = b / nbx, bx = b - by * nbx;
            const int x = (int)bx * 64 + lane, y0 = (int)by * R;
            uint32_t m[R];
#pragma unroll
            for (int r = 0; r < R; r++)
                m[r] = (x < a.W && y0 + r < a.H) ? (uint32_t)a.cells[(size_t)(y0 + r) * a.W + x] & 15u : 32u;
#pragma unroll
            for (int r = 0; r < R; r++) {
                const uint64_t q = __ballot(m[r] < 32u && ((a.airmask >> (m[r] & 31u)) & 1u));
                if (y0 + r < a.H && lane < 2) a.bits[(size_t)(y0 + r) * a.wpr + 2 * bx + lane] = (uint32_t)(q >> (32 * lane));
            }
        }
        for (uint32_t i = i0; i < a.bit_words; i += step) a.t[0].landed[i] = a.t[1].landed[i] = 0;
    }
    for (uint32_t i = i0; i < a.hcap; i += step)
        a.t[0].slots[i] = a.t[1].slots[i] = make_uint2(EMPTY, EMPTY);
    for (uint32_t i = i0; i < a.n; i += step) a.vkey[i] = -1;
    for (uint32_t i = i0; i < a.ncnt; i += step) a.cnt[i] = (i & 3u) == 1u ? 0xFFFFFFFFu : 0u;
    if (i0 < 2) a.totals[i0] = 0;
}

// An empty table for the cells' last writers.
__global__ void k_ph_clear(uint2 *slots, uint32_t cap) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < cap) slots[i] = make_uint2(EMPTY, 0u);
}

// Adds the landings of particles [0, n): key[i] is a cell or -1.  MAX keeps
// the highest index per cell (the last writer), else the lowest.
// prev: the counters of the round before (null: none); nothing to add if it
// changed no landing.
template <bool MAX>
__global__ void k_ph_insert(const int32_t *key, uint32_t n, Table t, uint32_t mask, int wpr, int W,
                            const uint32_t *prev) {
    if (prev && prev[0] == 0) return;
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    uint32_t *landed = t.landed;
    if (i >= n || key[i] < 0) return;
    const uint32_t c = (uint32_t)key[i];
    if (landed) {
        const uint32_t y = c / (uint32_t)W, x = c - y * (uint32_t)W;
        atomicOr(&landed[(size_t)y * wpr + (x >> 5)], 1u << (x & 31u));
    }
    for (uint32_t h = slot_of(c, mask);; h = (h + 1) & mask) {  // capacity >= 2n: a slot is always found
        const uint32_t old = atomicCAS(&t.slots[h].x, EMPTY, c);
        if (old == EMPTY || old == c) {
            if (MAX) atomicMax(&t.slots[h].y, i);
            else atomicMin(&t.slots[h].y, i);
            return;
        }
    }
}

__device__ __forceinline__ uint32_t ph_lookup(const uint2 *slots, uint32_t mask, uint32_t c) {
    for (uint32_t h = slot_of(c, mask);; h = (h + 1) & mask) {
        const uint2 q = slots[h];
        if (q.x == c) return q.y;
        if (q.x == EMPTY) return EMPTY;
    }
}

struct RoundArgs {
    const fsg_particle *p;  // the list as the pass found it
    PRes *res;
    int32_t *vkey;          // per particle: its non-air landing cell of the last round, or -1
    int32_t *wkey;          // per particle: its landing cell (any tile), or -1
    uint32_t n;
    const uint64_t *cells;
    int W, H;
    uint32_t airmask;
    int4 zone;
    uint32_t mask, hcap;    // of the tables
    Table view;             // the last round's landings (slots null: none)
    Table clear;            // the table before it, emptied here for the next round (slots null: it is empty)
    uint32_t *cnt;          // [0] landings that changed, [1] first particle whose landing changed,
                            // [2] cells appended to chg
    const uint32_t *prev;   // cnt of the last round (null: the first round)
    uint32_t *air_tiles;    // set if a particle landed with an air tile
    const int32_t *prev_chg;  // cells whose landing changed in the last round
    int32_t *chg;           // this round's changed cells
    AirMap am;
    BitMaps bm;
};

// One round: the particles from the first one whose landing changed against the
// grid and the view.  The round's kernels read the counters of the one before
// on the device, so several are enqueued at a time; after one that changed
// nothing the others end at once.  Bound by a lane's chain of loads and the
// search: 21 us for 40 000 particles on 4096^2, three rounds a pass (233 with
// the grid's own cells, and a look by the host after each).  A
// particle none of whose read cells changed its landing in the last round
// reads what it read then, so its outcome stands and it is not moved again.
constexpr uint32_t MAX_CHG = 4096;  // changed cells a round tests against (more: every particle moves)

template <bool BITS>
__global__ __launch_bounds__(256) void k_ph_round(RoundArgs a) {
    __shared__ uint32_t rows[BITS ? 32 * 256 : 1];
    __shared__ uint16_t firsts[BITS ? 32 * 256 : 1];
    __shared__ int2 cl[MAX_CHG];  // the changed cells as (x, y), staged once per workgroup
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    uint32_t start = 0;
    if (a.prev) {
        if (a.prev[0] == 0) return;
        start = a.prev[1];
    }
    if (a.clear.slots) {
        for (uint32_t h = i; h < a.hcap; h += gridDim.x * blockDim.x) {
            const uint32_t c = a.clear.slots[h].x;
            if (c == EMPTY) continue;
            if (a.clear.landed) {
                const uint32_t y = c / (uint32_t)a.W, x = c - y * (uint32_t)a.W;
                a.clear.landed[(size_t)y * a.bm.wpr + (x >> 5)] = 0;
            }
            a.clear.slots[h] = make_uint2(EMPTY, EMPTY);
        }
    }
    if (blockIdx.x * blockDim.x + blockDim.x <= start) return;
    // a long list of changes costs more to test than to move all
    if (a.prev && a.prev[2] <= MAX_CHG) {
        const uint32_t nchg = a.prev[2];
        for (uint32_t k = threadIdx.x; k < nchg; k += blockDim.x) {
            const int c = a.prev_chg[k];
            const int cy = c / a.W;
            cl[k] = make_int2(c - cy * a.W, cy);
        }
        __syncthreads();
        if (i >= a.n || i < start) return;
        const PRes &o = a.res[i];
        bool hit = false;
        if (o.bx0 <= o.bx1) {
            for (uint32_t k = 0; k < nchg; k++) {
                const int2 q = cl[k];
                hit |= q.x >= o.bx0 && q.x <= o.bx1 && q.y >= o.by0 && q.y <= o.by1;
            }
        }
        if (!hit) return;
    }
    if (i >= a.n || i < start) return;
    PState s;
    s.p = a.p[i];
    const View v{a.view.slots, a.mask, i};
    move_particle<BITS>(s, a.cells, a.W, a.H, a.airmask, a.zone, v, a.am, a.bm, rows + (BITS ? threadIdx.x : 0),
                        firsts + (BITS ? threadIdx.x : 0));
    PRes r;
    r.p = s.p;
    r.kind = s.kind;
    r.land = s.land;
    r.bx0 = s.bx0;
    r.by0 = s.by0;
    r.bx1 = s.bx1;
    r.by1 = s.by1;
    a.res[i] = r;
    const bool solid = s.kind == 2 && !((a.airmask >> (uint32_t)(s.p.tile.mat & 15u)) & 1u);
    if (s.kind == 2 && !solid) *a.air_tiles = 1u;
    const int32_t k = solid ? s.land : -1;
    const int32_t old = a.vkey[i];
    if (k != old) {
        atomicAdd(&a.cnt[0], 1u);
        atomicMin(&a.cnt[1], i);
        a.vkey[i] = k;
        const uint32_t at = atomicAdd(&a.cnt[2], (old >= 0 ? 1u : 0u) + (k >= 0 ? 1u : 0u));
        uint32_t o2 = at;
        if (old >= 0) a.chg[o2++] = old;
        if (k >= 0) a.chg[o2] = k;
    }
    a.wkey[i] = s.kind == 2 ? s.land : -1;
}

struct ApplyArgs {
    fsg_particle *p;
    const PRes *res;
    uint8_t *alive;
    uint32_t n;             // particles [0, n) are final
    uint64_t *cells;
    int W, H, tiles_x;
    uint32_t *flags;
    const uint2 *slots;     // last writer per landing cell (null: a cell has one)
    uint32_t mask;
    unsigned long long *landed;
    uint32_t *blk;          // survivors per block of 1024 particles (null: not counted)
};

// Final outcomes.  A cell that a particle with a tile other than air lands in
// is free to none after it, so cells have one writer unless air tiles
// landed: then the last one writes.
__global__ __launch_bounds__(1024) void k_ph_apply(ApplyArgs a) {
    __shared__ uint32_t wsum[16];
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    bool keep = false;
    unsigned long long nl = 0;
    if (i < a.n) {
        const PRes r = a.res[i];
        if (r.kind == 2) {
            nl = 1;
            if (!a.slots || ph_lookup(a.slots, a.mask, (uint32_t)r.land) == i) {
                const fsg_cell &tl = r.p.tile;
                a.cells[r.land] = (uint64_t)tl.mat | ((uint64_t)(uint16_t)tl.temp << 16) | ((uint64_t)tl.rgba << 32);
                if (a.flags) {
                    const int cy = r.land / a.W, cx = r.land - cy * a.W;
                    atomicOr(&a.flags[(cy / fsg::TH) * a.tiles_x + cx / fsg::TW], fsg::F_WAKE_ALL);
                }
            }
        }
        keep = r.kind == 0 && !(r.p.y > (float)a.H);  // erase_if(y > height), world.cpp:2190
        a.alive[i] = keep;
        if (r.kind == 0) a.p[i] = r.p;
    }
    for (int off = 32; off > 0; off >>= 1) nl += __shfl_xor(nl, off, 64);
    if ((threadIdx.x & 63) == 0 && nl) atomicAdd(a.landed, nl);
    if (!a.blk) return;
    const uint64_t m = __ballot(keep);
    if ((threadIdx.x & 63) == 0) wsum[threadIdx.x >> 6] = (uint32_t)__popcll(m);
    __syncthreads();
    if (threadIdx.x == 0) {
        uint32_t t = 0;
        for (int k = 0; k < 16; k++) t += wsum[k];
        a.blk[blockIdx.x] = t;
    }
}

// ---- survivors in list order ---------------------------------------------------
// Counts per 1024-particle block (from k_ph_apply, or k_pc_count where the
// batch walk ended the pass), then each block writes its survivors from its
// offset: the sum of the counts before it, which it makes itself for up to
// 1024 blocks; above, one workgroup scans the counts first.
__global__ __launch_bounds__(1024) void k_pc_count(const uint8_t *alive, uint32_t n, uint32_t *blk) {
    __shared__ uint32_t wsum[16];
    const uint32_t i = blockIdx.x * 1024 + threadIdx.x;
    const uint64_t m = __ballot(i < n && alive[i]);
    if ((threadIdx.x & 63) == 0) wsum[threadIdx.x >> 6] = (uint32_t)__popcll(m);
    __syncthreads();
    if (threadIdx.x == 0) {
        uint32_t t = 0;
        for (int k = 0; k < 16; k++) t += wsum[k];
        blk[blockIdx.x] = t;
    }
}

__global__ __launch_bounds__(1024) void k_pc_scan(uint32_t *blk, uint32_t nb, uint32_t *total) {
    __shared__ uint32_t part[1024];
    __shared__ uint32_t carry;
    if (threadIdx.x == 0) carry = 0;
    __syncthreads();
    for (uint32_t b0 = 0; b0 < nb; b0 += 1024) {
        const uint32_t i = b0 + threadIdx.x;
        const uint32_t v = i < nb ? blk[i] : 0u;
        part[threadIdx.x] = v;
        __syncthreads();
        for (uint32_t off = 1; off < 1024; off <<= 1) {  // inclusive Hillis-Steele scan
            const uint32_t add = threadIdx.x >= off ? part[threadIdx.x - off] : 0u;
            __syncthreads();
            part[threadIdx.x] += add;
            __syncthreads();
        }
        if (i < nb) blk[i] = carry + part[threadIdx.x] - v;
        __syncthreads();
        if (threadIdx.x == 0) carry += part[1023];
        __syncthreads();
    }
    if (threadIdx.x == 0) *total = carry;
}

__global__ __launch_bounds__(1024) void k_pc_scatter(const fsg_particle *in, const uint8_t *alive, uint32_t n,
                                                     const uint32_t *blk, bool scanned, fsg_particle *out,
                                                     uint32_t *total) {
    __shared__ uint32_t wsum[16], before[16];
    const uint32_t i = blockIdx.x * 1024 + threadIdx.x;
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    const bool keep = i < n && alive[i];
    const uint64_t m = __ballot(keep);
    if (lane == 0) wsum[wv] = (uint32_t)__popcll(m);
    if (!scanned) {
        uint32_t v = threadIdx.x < blockIdx.x ? blk[threadIdx.x] : 0u;
        for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
        if (lane == 0) before[wv] = v;
    }
    __syncthreads();
    uint32_t off = scanned ? blk[blockIdx.x] : 0u;
    if (!scanned)
        for (int k = 0; k < 16; k++) off += before[k];
    for (int k = 0; k < wv; k++) off += wsum[k];
    if (keep) out[off + __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u))] = in[i];
    if (!scanned && blockIdx.x == gridDim.x - 1 && threadIdx.x == 1023) *total = off + wsum[15];
}

using fsg_impl::dev_alloc;
using fsg_impl::dev_free;

// Grows the list buffers to hold `want` particles, keeping the list.
int grow_lists(fsg_world *w, size_t want) {
    if (w->part_cap >= want) return FSG_OK;
    fsg_ctx *c = w->ctx;
    const size_t nc = std::max(want, w->part_cap * 2);
    void *a = nullptr, *b = nullptr, *f = nullptr;
    if (dev_alloc(c, &a, nc * sizeof(fsg_particle))) return FSG_ERR_NOMEM;
    if (dev_alloc(c, &b, nc * sizeof(fsg_particle))) {
        dev_free(a);
        return FSG_ERR_NOMEM;
    }
    if (dev_alloc(c, &f, nc)) {
        dev_free(a);
        dev_free(b);
        return FSG_ERR_NOMEM;
    }
    if (w->npart) HIPCHK(hipMemcpyAsync(a, w->d_part, w->npart * sizeof(fsg_particle), hipMemcpyDeviceToDevice, c->stream));
    dev_free(w->d_part);
    dev_free(w->d_part2);
    dev_free(w->d_part_alive);
    w->d_part = static_cast<fsg_particle *>(a);
    w->d_part2 = static_cast<fsg_particle *>(b);
    w->d_part_alive = static_cast<uint8_t *>(f);
    w->part_cap = nc;
    return FSG_OK;
}

// Rounds before a list whose landings keep changing goes to the batch walk: as
// many as the walk would need batches for the list, as a round and a batch
// take about the same time and a round moves every particle (300 000 on 1024^2,
// most of them in packed heaps: 133 ms a pass with 24 rounds, 9 with 256;
// 20 heaps of 150 particles: 12 ms with 24, 59 with 256).  Three are enqueued
// before the host looks at their counters, then six at a time (a spray over
// terrain takes three; a round that has nothing to do costs about 5 us, a
// look 20).
constexpr int MAX_ROUNDS = 256, MIN_ROUNDS = 24;
constexpr int ROUNDS_AHEAD = 3, LATER_AHEAD = 6;
constexpr uint32_t CNT_WORDS = 4 * MAX_ROUNDS + 4;  // four a round, then: air tiles landed

// Round buffers for `n` particles, carved from one block: results, the two
// landing keys, the compaction's block offsets, counters, and two landing
// tables (capacity the power of two >= 2n, so they are at most half full).
struct RoundBufs {
    PRes *res;
    int32_t *vkey, *wkey, *chg[2];
    uint32_t *blk, *cnt, *air;
    Table t[2];
    uint32_t hcap, air_words;
    int air_wpr;
    uint32_t *bits;  // the grid's air plane (null: not built), of bit_words, as each table's
    uint32_t bit_words;
    int bit_wpr;
};

size_t align256(size_t v) { return (v + 255) & ~(size_t)255; }

// The planes' build reads the whole grid (22 us for 4096^2) and the passes they
// are for are bounded by one lane's chain of loads whatever their number, so
// up to 2^25 cells they are always built (a pass of 10 particles on 4096^2
// took 206 us with the on-demand map, of 1000 745; with the planes and the
// launches below 84 and 115), and above for one particle per 2^17 cells, from
// where they are ahead everywhere.  us a pass, planes / map, over ground: 8192^2
// 200 particles 201 / 247, 400 208 / 492; 16384 x 8192 200 316 / 253, 800 329 /
// 676; 16384^2 800 563 / 599, 3000 576 / 744; in the air 8192^2 200 183 / 130, 400
// 196 / 332; 16384 x 8192 200 301 / 127, 400 311 / 338; 16384^2 1500 546 / 456,
// 3000 552 / 584.
bool want_planes(const fsg_world *w, size_t n) {
    const size_t cells = (size_t)w->d.W * w->d.H;
    return cells <= (size_t)1 << 25 || n >= cells >> 17;
}

int round_bufs(fsg_world *w, size_t n, RoundBufs &b) {
    uint32_t hcap = 1024;
    while (hcap < 2 * n) hcap <<= 1;
    const size_t nb = n / 1024 + 2;
    const int nbx = (w->d.W + 7) / 8, nby = (w->d.H + 7) / 8;
    b.air_wpr = (nbx + 15) / 16;
    b.air_words = (uint32_t)((size_t)b.air_wpr * nby);
    b.bit_wpr = 2 * ((w->d.W + 63) / 64);
    bool planes = want_planes(w, n);
    b.bit_words = planes ? (uint32_t)((size_t)b.bit_wpr * w->d.H) : 0u;
    size_t sz = align256(n * sizeof(PRes)) + 2 * align256(n * 4) + 2 * align256(n * 8) + align256(nb * 4) +
                align256(CNT_WORDS * 4) + 2 * align256((size_t)hcap * 8) + align256((size_t)b.air_words * 4) +
                3 * align256((size_t)b.bit_words * 4);
    if (w->pround_cap < sz) {
        void *q = nullptr;
        int rc = dev_alloc(w->ctx, &q, sz);
        if (rc && planes) {  // short of memory: without the planes
            planes = false;
            sz -= 3 * align256((size_t)b.bit_words * 4);
            b.bit_words = 0;
            rc = w->pround_cap < sz ? dev_alloc(w->ctx, &q, sz) : FSG_OK;
        }
        if (rc) return FSG_ERR_NOMEM;
        if (q) {
            dev_free(w->d_pround);
            w->d_pround = q;
            w->pround_cap = sz;
        }
    }
    char *c = static_cast<char *>(w->d_pround);
    b.res = reinterpret_cast<PRes *>(c);
    c += align256(n * sizeof(PRes));
    b.vkey = reinterpret_cast<int32_t *>(c);
    c += align256(n * 4);
    b.wkey = reinterpret_cast<int32_t *>(c);
    c += align256(n * 4);
    for (int k = 0; k < 2; k++) {  // each particle adds at most two cells per round
        b.chg[k] = reinterpret_cast<int32_t *>(c);
        c += align256(n * 8);
    }
    b.blk = reinterpret_cast<uint32_t *>(c);
    c += align256(nb * 4);
    b.cnt = reinterpret_cast<uint32_t *>(c);
    c += align256(CNT_WORDS * 4);
    for (Table &t : b.t) {
        t.slots = reinterpret_cast<uint2 *>(c);
        c += align256((size_t)hcap * 8);
    }
    b.air = reinterpret_cast<uint32_t *>(c);
    c += align256((size_t)b.air_words * 4);
    uint32_t *plane[3];
    for (uint32_t *&q : plane) {
        q = planes ? reinterpret_cast<uint32_t *>(c) : nullptr;
        c += align256((size_t)b.bit_words * 4);
    }
    b.bits = plane[0];
    b.t[0].landed = plane[1];
    b.t[1].landed = plane[2];
    b.hcap = hcap;
    return FSG_OK;
}

}  // namespace

extern "C" int fsg_world_particles_add(fsg_world *w, const fsg_particle *p, size_t n) {
    if (!w || (n && !p)) return FSG_ERR_INVALID;
    for (size_t i = 0; i < n; i++) {
        const uint16_t m = p[i].tile.mat;
        if ((m & 0xFE00u) || (uint32_t)(m & 0xFFu) >= w->cfg.n_materials) return FSG_ERR_INVALID;
        if (!std::isfinite(p[i].x) || !std::isfinite(p[i].y) || !std::isfinite(p[i].vx) || !std::isfinite(p[i].vy) ||
            !std::isfinite(p[i].ax) || !std::isfinite(p[i].ay) || !std::isfinite(p[i].target_x) ||
            !std::isfinite(p[i].target_y) || !std::isfinite(p[i].target_force) || p[i].in_object_state > 2 ||
            (p[i].flags & ~(FSG_PARTICLE_PHASE | FSG_PARTICLE_TEMPORARY)))
            return FSG_ERR_INVALID;
    }
    if (n == 0) return FSG_OK;
    if (w->npart + n > 0xFFFFFFFFull) return FSG_ERR_INVALID;
    fsg_ctx *c = w->ctx;
    HIPCHK(hipSetDevice(c->device));
    if (int rc = grow_lists(w, w->npart + n)) return rc;
    if (int rc = fsg_impl::copy_in(c, w->d_part + w->npart, p, n * sizeof(fsg_particle))) return rc;
    w->npart += n;
    return FSG_OK;
}

extern "C" int fsg_world_particles_tick(fsg_world *w, size_t *alive, size_t *landed) {
    if (!w) return FSG_ERR_INVALID;
    fsg_ctx *c = w->ctx;
    HIPCHK(hipSetDevice(c->device));
    const uint32_t n = (uint32_t)w->npart;
    unsigned long long nl = 0;
    if (n) {
        if (!w->d_part_cnt) {
            void *q = nullptr;
            if (dev_alloc(c, &q, 16)) return FSG_ERR_NOMEM;
            w->d_part_cnt = static_cast<unsigned long long *>(q);
        }
        RoundBufs b;
        if (int rc = round_bufs(w, n, b)) return rc;
        hipStream_t st = c->stream;
        uint32_t airmask = 0;
        for (uint32_t m = 0; m < w->cfg.n_materials; m++)
            if (w->cfg.materials[m].type == FSG_AIR) airmask |= 1u << m;
        const int4 zone = make_int4(w->d.zx0, w->d.zy0, w->d.zx1, w->d.zy1);
        uint64_t *cells = w->d.buf[w->d.tick & 1];
        // landings wake their chunks for the next tick (no flags: it processes every chunk)
        uint32_t *flags = w->flags_valid ? w->d.flags[(w->d.tick + 1) & 1] : nullptr;
        const unsigned ng = (n + 255) / 256;
        {
            PrepArgs pa{cells, w->d.W, w->d.H, airmask, b.bits, b.bit_wpr, b.bit_words, b.hcap, n, CNT_WORDS,
                        {b.t[0], b.t[1]}, b.vkey, b.cnt, w->d_part_cnt};
            // a workgroup per four wave tiles of the plane, up to 16 a CU
            const size_t tiles = b.bits ? (size_t)(b.bit_wpr / 2) * ((w->d.H + 7) / 8) : 0;
            const size_t g = std::max<size_t>((tiles + 3) / 4, std::max<size_t>(ng, b.hcap / 256));
            k_ph_prep<<<(unsigned)std::min<size_t>(g, (size_t)c->n_cu * 16), 256, 0, st>>>(pa);
        }
        const unsigned ag = (b.air_words + 255) / 256;
        if (!b.bits) k_u32_fill<<<ag, 256, 0, st>>>(b.air, b.air_words, 0u);
        uint32_t final_n = 0;  // particles [0, final_n) have their outcomes
        uint32_t h[CNT_WORDS];
        // the walk's time is at least that of its batches, so rounds may take as many
        const int most = (int)std::min<size_t>(MAX_ROUNDS, std::max<size_t>(MIN_ROUNDS, n / PT));
        for (int round = 0; round < most && final_n < n;) {
            const int first = round;
            for (; round < std::min(first + (first ? LATER_AHEAD : ROUNDS_AHEAD), most); round++) {
                RoundArgs ra{};
                ra.p = w->d_part;
                ra.res = b.res;
                ra.vkey = b.vkey;
                ra.wkey = b.wkey;
                ra.n = n;
                ra.cells = cells;
                ra.W = w->d.W;
                ra.H = w->d.H;
                ra.airmask = airmask;
                ra.zone = zone;
                ra.mask = b.hcap - 1;
                ra.hcap = b.hcap;
                ra.cnt = b.cnt + 4 * round;
                ra.air_tiles = b.cnt + 4 * MAX_ROUNDS;
                ra.prev_chg = b.chg[(round + 1) & 1];
                ra.chg = b.chg[round & 1];
                ra.am = AirMap{b.air, b.air_wpr};
                ra.bm = BitMaps{b.bits, nullptr, b.bit_wpr};
                if (round > 0) {
                    ra.prev = ra.cnt - 4;
                    ra.view = b.t[round & 1];
                    ra.bm.landed = ra.view.landed;
                    if (round > 1) ra.clear = b.t[(round + 1) & 1];
                    k_ph_insert<false><<<ng, 256, 0, st>>>(b.vkey, n, ra.view, ra.mask, b.bit_wpr, w->d.W, ra.prev);
                }
                if (b.bits) k_ph_round<true><<<ng, 256, 0, st>>>(ra);
                else k_ph_round<false><<<ng, 256, 0, st>>>(ra);
            }
            HIPCHK(hipGetLastError());
            if (int rc = fsg_impl::copy_out(c, {{h, b.cnt, sizeof h}})) return rc;
            for (int r = first; r < round && final_n < n; r++)
                // no landing changed: every outcome is the sequential one; else
                // the particles before the first changed landing are final
                final_n = h[4 * r] == 0 ? n : h[4 * r + 1];
        }
        if (final_n > 0) {
            ApplyArgs aa{w->d_part, b.res, w->d_part_alive, final_n, cells, w->d.W, w->d.H, w->d.tiles_x, flags,
                         nullptr, b.hcap - 1, w->d_part_cnt, final_n == n ? b.blk : nullptr};
            if (h[4 * MAX_ROUNDS]) {  // air tiles: the last particle landing in a cell writes it
                const Table t{b.t[0].slots, nullptr};
                k_ph_clear<<<(b.hcap + 255) / 256, 256, 0, st>>>(t.slots, b.hcap);
                k_ph_insert<true><<<(final_n + 255) / 256, 256, 0, st>>>(b.wkey, final_n, t, b.hcap - 1, 0, w->d.W,
                                                                         nullptr);
                aa.slots = t.slots;
            }
            k_ph_apply<<<(final_n + 1023) / 1024, 1024, 0, st>>>(aa);
        }
        if (final_n < n) {
            // the rest, in order, by the batch walk over the grid the prefix left
            PArgs a;
            a.p = w->d_part;
            a.alive = w->d_part_alive;
            a.start = final_n;
            a.n = n;
            a.cells = cells;
            a.W = w->d.W;
            a.H = w->d.H;
            a.tiles_x = w->d.tiles_x;
            a.zone = zone;
            a.airmask = airmask;
            a.flags = flags;
            a.landed = w->d_part_cnt;
            a.airbits = b.air;
            a.air_wpr = b.air_wpr;
            if (b.bits) k_u32_fill<<<ag, 256, 0, st>>>(b.air, b.air_words, 0u);
            k_particles<<<1, PT, 0, st>>>(a);
        }
        const uint32_t nb = (n + 1023) / 1024;
        uint32_t *total = reinterpret_cast<uint32_t *>(w->d_part_cnt + 1);
        if (final_n < n) k_pc_count<<<nb, 1024, 0, st>>>(w->d_part_alive, n, b.blk);
        if (nb > 1024) k_pc_scan<<<1, 1024, 0, st>>>(b.blk, nb, total);
        k_pc_scatter<<<nb, 1024, 0, st>>>(w->d_part, w->d_part_alive, n, b.blk, nb > 1024, w->d_part2, total);
        HIPCHK(hipGetLastError());
        unsigned long long sums[2] = {0, 0};
        if (int rc = fsg_impl::copy_out(c, {{sums, w->d_part_cnt, 16}})) return rc;
        nl = sums[0];
        std::swap(w->d_part, w->d_part2);  // the survivors, in order, are the list
        w->npart = (size_t)(uint32_t)sums[1];
    }
    if (alive) *alive = w->npart;
    if (landed) *landed = (size_t)nl;
    return FSG_OK;
}

extern "C" int fsg_world_particles_get(fsg_world *w, fsg_particle *out, size_t cap, size_t *n) {
    if (!w || (cap && !out)) return FSG_ERR_INVALID;
    fsg_ctx *c = w->ctx;
    HIPCHK(hipSetDevice(c->device));
    const size_t k = std::min(cap, w->npart);
    if (k)
        if (int rc = fsg_impl::copy_out(c, {{out, w->d_part, k * sizeof(fsg_particle)}})) return rc;
    if (n) *n = w->npart;
    return FSG_OK;
}
