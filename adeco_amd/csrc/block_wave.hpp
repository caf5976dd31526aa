// Wavefront machinery of the block deposits (blocks.hip, direct.hip): how a tet's covered cells are cut
// into blocks, the per-wave work queues, and the loop that clips them.
//
// A block to clip is queued by its work class and a queue that holds 64 of them is clipped by the whole
// wave: each lane cuts its own block's tet, and the pieces (leaves) are gathered over the lanes and summed one
// per lane, each into its block's LDS column (LeafQueue).  A cell whose share is small against the rounding of
// the differences goes to one more queue, whose passes recompute it alone.
#pragma once

#include <hip/hip_runtime.h>

#include "batched_impl.hpp"
#include "block_clip.hpp"
#include "wave_tiles.hpp"

namespace adeco {

constexpr int kClasses = 8;            // queues of blocks to clip
constexpr int kExact = kClasses;       // the queue of single cells to recompute
constexpr int kQueues = kClasses + 1;
static_assert(kClasses <= 8 && kQueues <= 16, "the drain's prefix sum and the counts");

// Per-wavefront LDS.  A queue entry is an int2 that the kernel's loader
// understands.  An entry that finds its queue full is carried per lane and takes its place once that
// queue has been clipped; qn[b] counts queue b's entries and its carried ones.
struct BlockLds {
    int qn[16];
    int2 q[kQueues][kWaveTile];
    int2 carry[kWaveTile];
    signed char carry_key[kWaveTile];
    unsigned char cell[kWaveTile];  // of each exact-queue entry
    double leaf[5][kWaveTile];      // leaves of the pass: 4 heights and the share,
    unsigned leaf_to[kWaveTile];    // and where they count
    union {
        unsigned long long sum[kBlockCells][kWaveTile];  // each lane's shares, in units of 2^-62
        double keep[15][kWaveTile];             // each lane's storage of a recompute
        int mark[kWaveTile];       // starts of the tile being classified
    };
};

// How covered cells are cut into blocks: blocks of b cells, n of them, per axis (x, y, z in the pair's
// order, extents ex <= ey <= ez).  A cover of at most kBlockCells cells is one block; else x keeps up to 2 cells,
// z up to 6 (more where x and y have few) and y what is left, the cells spread evenly over an axis' blocks.
// Large blocks cut fewer faces between blocks, and planes across z cost least.  24 cells are what the LDS of a
// wave holds; against 16 (2 x 2 x 4): 15.3 M pairs on 16^3-cell leaves 4.02 -> 3.71 ms, 6.7 M pairs on
// 32^3-cell leaves 10.9 -> 9.75, a 64^3 request on a 128^3 lattice 515 -> 409 us.
struct BlockShape {
    int b[3], n[3];
};

__device__ __forceinline__ BlockShape block_shape(int ex, int ey, int ez) {
    static_assert(kBlockCells == 24, "block sizes");
    const int e[3] = {ex, ey, ez};
    BlockShape s;
    for (int a = 0; a < 3; ++a) {
        s.b[a] = e[a];
        s.n[a] = 1;
    }
    if (ex * ey * ez <= kBlockCells) return s;
    const auto cut = [&](int a, int most) {
        if (e[a] <= most) return;
        const int n = int(udiv_small(unsigned(e[a] + most - 1), unsigned(most)));
        s.b[a] = int(udiv_small(unsigned(e[a] + n - 1), unsigned(n)));
        s.n[a] = int(udiv_small(unsigned(e[a] + s.b[a] - 1), unsigned(s.b[a])));
    };
    cut(0, 2);
    const int xy = s.b[0] * min(ey, 4);
    cut(2, xy == 1 ? 24 : (xy == 2 ? 12 : (xy == 3 ? 8 : 6)));
    // 24 / (x * z): the quotient is at least 0.02 from the next whole number
    cut(1, int(24.5f * __builtin_amdgcn_rcpf(float(s.b[0] * s.b[2]))));
    return s;
}

// Axis order of a cover, packed in 3 bits: the axis of z and whether x and y are the next two axes in
// cyclic order or the reverse.
__device__ __forceinline__ int role_axis(int code, int role) {
    const int za = code & 3, u = za == 2 ? 0 : za + 1, v = u == 2 ? 0 : u + 1;
    const bool swap = code & 4;
    return role == 2 ? za : ((role == 0) != swap ? u : v);
}

template <class T>
__device__ __forceinline__ T pick(int a, T v0, T v1, T v2) {
    return a == 0 ? v0 : (a == 1 ? v1 : v2);
}

// The order of the axes for extents e: z the longest (ties: z, then y), x the shorter of the others.
__device__ __forceinline__ int role_code(const int e[3]) {
    const int za = e[2] >= e[1] && e[2] >= e[0] ? 2 : (e[1] >= e[0] ? 1 : 0);
    const int u = za == 2 ? 0 : za + 1, w = u == 2 ? 0 : u + 1;
    return za | (pick(w, e[0], e[1], e[2]) < pick(u, e[0], e[1], e[2]) ? 4 : 0);
}

// Covered cells l..h of one axis for a tet between mn and mx (in cells from the grid's face): the cells
// whose box it can strictly overlap, widened by 1e-9 of a cell and kept inside the grid.
__device__ __forceinline__ void covered(double mn, double mx, int dims, int& l, int& h) {
    const double top = double(dims - 1);
    l = int(fmax(fmin(floor(mn - 1e-9), top), 0.0));
    h = int(fmax(fmin(floor(mx + 1e-9), top), 0.0));
}

// A block of a cover: its corner cell (in the cover's axis order), its sizes and the tet's vertices from
// the corner.
struct Block {
    int lo[3], c[3];
    double x[4], y[4], z[4];
};

// lo, e: the cover's first cell and extents in its axis order; s: the vertices in cells, in that order.
__device__ __forceinline__ Block make_block(const int lo[3], const int e[3], const double s[4][3], unsigned unit) {
    Block b;
    const BlockShape sh = block_shape(e[0], e[1], e[2]);
    int i[3] = {0, 0, 0};
    if (unit) {
        const unsigned rest = sh.n[2] == 1 ? unit : udiv_small(unit, unsigned(sh.n[2]));
        i[2] = int(unit - rest * unsigned(sh.n[2]));
        i[0] = sh.n[1] == 1 ? int(rest) : int(udiv_small(rest, unsigned(sh.n[1])));
        i[1] = int(rest) - i[0] * sh.n[1];
    }
    for (int a = 0; a < 3; ++a) {
        b.lo[a] = lo[a] + i[a] * sh.b[a];
        b.c[a] = min(sh.b[a], e[a] - i[a] * sh.b[a]);
    }
    for (int q = 0; q < 4; ++q) {
        b.x[q] = s[q][0] - double(b.lo[0]);
        b.y[q] = s[q][1] - double(b.lo[1]);
        b.z[q] = s[q][2] - double(b.lo[2]);
    }
    return b;
}

// Where a block's cells lie: the offset of its first cell and the strides of its axes.
struct Place {
    int64_t corner, sx, sy, sz;
};

__device__ __forceinline__ Place place_of(const int lo[3], int code, int dims) {
    const int64_t s1 = dims, s2 = int64_t(dims) * dims;
    Place p;
    p.sx = pick(role_axis(code, 0), int64_t(1), s1, s2);
    p.sy = pick(role_axis(code, 1), int64_t(1), s1, s2);
    p.sz = pick(role_axis(code, 2), int64_t(1), s1, s2);
    p.corner = lo[0] * p.sx + lo[1] * p.sy + lo[2] * p.sz;
    return p;
}

// Visits the cells of a block in the order of its shares: f(index, offset in the grid).
template <class F>
__device__ __forceinline__ void for_cells(const int c[3], const Place& p, F f) {
    const int n = c[0] * c[1] * c[2];
    int b = 0, k = 0;
    int64_t at = p.corner;
    const int64_t next_y = p.sy - c[2] * p.sz, next_x = p.sx - c[1] * p.sy;
    for (int i = 0; i < n; ++i) {
        f(i, at);
        at += p.sz;
        if (++k == c[2]) {
            k = 0;
            at += next_y;
            if (++b == c[1]) {
                b = 0;
                at += next_x;
            }
        }
    }
}

// Work class of a block to clip: by the pieces that the x planes leave of the tet (1 for each plane with 1 or 3
// vertices below, else 3), and where they are few by the planes that cut it across y.  The class only groups
// blocks of similar loops (8 classes against 6 by the planes alone: 9.75 -> 9.2 ms for the large tets above,
// 3.71 -> 3.68 for the small ones).  mn, mx: the tet's extents from the block's corner.
__device__ __forceinline__ int work_class(const Block& b, const double mn[3], const double mx[3]) {
    const int fx = floor_clamped(mn[0], b.c[0]) + 1, lx = min(ceil_clamped(mx[0], b.c[0]) - 1, b.c[0]);
    const int fy = floor_clamped(mn[1], b.c[1]) + 1, ly = min(ceil_clamped(mx[1], b.c[1]) - 1, b.c[1]);
    const int py = ly - fy + 1;
    int pieces = 0;
    for (int p = 0; p <= 2; ++p) {  // (a block has at most 2 cells across x)
        const int n = int(b.x[0] < double(p)) + int(b.x[1] < double(p)) + int(b.x[2] < double(p)) + int(b.x[3] < double(p));
        pieces += p >= fx && p <= lx ? (n == 2 ? 3 : 1) : 0;
    }
    if (pieces <= 1) return 2 * pieces + int(py > pieces);
    if (pieces == 3) return 5 + int(py > 1);
    return pieces == 2 ? 4 : 7;
}

enum BlockClass : int { kBlockEmpty = -1, kBlockTet = -2, kBlockFull = -3 };

// What to do with a block: nothing, deposit the whole tet in its only cell, fill it, or clip it (the work
// class >= 0).  The tet is positively oriented in the block's axis order.
__device__ __forceinline__ int classify_block(const Block& b) {
    const double mn[3] = {fmin(fmin(b.x[0], b.x[1]), fmin(b.x[2], b.x[3])), fmin(fmin(b.y[0], b.y[1]), fmin(b.y[2], b.y[3])),
                          fmin(fmin(b.z[0], b.z[1]), fmin(b.z[2], b.z[3]))};
    const double mx[3] = {fmax(fmax(b.x[0], b.x[1]), fmax(b.x[2], b.x[3])), fmax(fmax(b.y[0], b.y[1]), fmax(b.y[2], b.y[3])),
                          fmax(fmax(b.z[0], b.z[1]), fmax(b.z[2], b.z[3]))};
    const double box[3] = {double(b.c[0]), double(b.c[1]), double(b.c[2])};
    bool hit = true, inside = true;
    for (int a = 0; a < 3; ++a) {
        hit = hit && mn[a] < box[a] && 0.0 < mx[a];
        inside = inside && mn[a] >= 0.0 && mx[a] <= box[a];
    }
    if (!hit) return kBlockEmpty;
    if (inside) {
        if (b.c[0] * b.c[1] * b.c[2] == 1) return kBlockTet;
    } else {
        V3<double> s[4];
        for (int q = 0; q < 4; ++q) s[q] = mk(b.x[q], b.y[q], b.z[q]);
        const int cls = classify_margin(s, box);
        if (cls == CLS_NONE) return kBlockEmpty;
        if (cls == CLS_CELL_IN_TET) return kBlockFull;
    }
    return work_class(b, mn, mx);
}

// set bits of m below this lane
__device__ __forceinline__ int mbcnt64(unsigned long long m) {
    return int(__builtin_amdgcn_mbcnt_hi(unsigned(m >> 32), __builtin_amdgcn_mbcnt_lo(unsigned(m), 0u)));
}

// Appends each lane's entry to queue `key` (none when key < 0).  Every queue holds < 64 entries before,
// so a count reaches at most 127; an entry beyond 64 is carried.
__device__ __forceinline__ void push_blocks(BlockLds& L, int lane, int key, int2 entry) {
    int ckey = -1;
    if (key >= 0) {
        const int pos = atomicAdd(&L.qn[key], 1);
        if (pos < kWaveTile) {
            L.q[key][pos] = entry;
        } else {
            ckey = key;
            L.carry[lane] = entry;
        }
    }
    L.carry_key[lane] = (signed char)ckey;
    wave_sync();
}

// A lane's column of shares, summed as integers of 2^-62: leaves reach it in an order that depends on what else
// the wave clips, and a sum of integers does not depend on its order (the unit is far below the rounding of a
// share, and what wraps on the way wraps back).
struct LaneShares {
    unsigned long long* a;
    __device__ __forceinline__ static long long term(double share) {
        const double t = share * 0x1p30, hi = floor(t);
        return (long long)((unsigned long long)(unsigned)int(hi) << 32 | unsigned((t - hi) * 0x1p32));
    }
    __device__ __forceinline__ static double value(unsigned long long v) { return double((long long)v) * 0x1p-62; }
    __device__ __forceinline__ void add(int i, long long v) {
        __hip_atomic_fetch_add(a + i * kWaveTile, (unsigned long long)v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    }
};

// Leaves of a pass' blocks, gathered over the lanes and summed 64 at a time, one per lane.  Half of a block's
// work is its leaves, and their number differs much from block to block (2-40): summed in the loops that make
// them, on average a quarter of the lanes had one (large tets; 45 M blocks on 32^3-cell leaves 15.3 ms against
// 10.8, 196 608 tets on 64^3 cells 430 us against 314; one-block tets, of 3 leaves each, 4.26 ms against 4.02
// for 15.3 M pairs).
struct LeafQueue {
    BlockLds& L;
    int lane;
    int n = 0;  // leaves waiting, < 64
    __device__ __forceinline__ bool any(bool b) const { return __ballot(b) != 0ull; }
    __device__ __forceinline__ void put(int at, double z0, double z1, double z2, double z3, double w, Target t) {
        L.leaf[0][at] = z0;
        L.leaf[1][at] = z1;
        L.leaf[2][at] = z2;
        L.leaf[3][at] = z3;
        L.leaf[4][at] = w;
        L.leaf_to[at] = unsigned(lane) | unsigned(t.base) << 6 | unsigned(t.dy) << 11 | unsigned(t.dx) << 16 | unsigned(t.cz) << 21;
    }
    __device__ __forceinline__ void sum(int count) {
        wave_sync();
        if (lane < count) {
            const unsigned to = L.leaf_to[lane];
            Target t;
            t.base = int(to >> 6) & 31;
            t.dy = int(to >> 11) & 31;
            t.dx = int(to >> 16) & 31;
            t.cz = int(to >> 21);
            LaneShares acc{&L.sum[0][to & 63u]};
            block_leaf(L.leaf[0][lane], L.leaf[1][lane], L.leaf[2][lane], L.leaf[3][lane], L.leaf[4][lane], t, acc);
        }
        wave_sync();
    }
    __device__ __forceinline__ void leaf(bool on, double z0, double z1, double z2, double z3, double w, Target t) {
        const unsigned long long m = __ballot(on);
        const int at = n + mbcnt64(m);
        if (on && at < kWaveTile) put(at, z0, z1, z2, z3, w, t);
        n += int(__popcll(m));
        if (n >= kWaveTile) {
            sum(kWaveTile);
            if (on && at >= kWaveTile) put(at - kWaveTile, z0, z1, z2, z3, w, t);
            n -= kWaveTile;
        }
    }
};

// Clips each lane's queued block (where on) and deposits its cells, except those whose share is small against
// the rounding of the differences: returns their mask (bit = index of the cell in the block).
// Loader: block(entry) the block, place(entry, lo) the place of a cell of it in its grid (looked up again
// after the clip, which needs the registers), add(entry, offset, share) the deposit.
template <class Loader>
__device__ __forceinline__ unsigned clip_blocks(const Loader& ld, bool on, int2 e, const Block& b, BlockLds& L, int lane) {
    unsigned long long* sum = &L.sum[0][lane];
    for (int i = 0; i < kBlockCells; ++i) sum[i * kWaveTile] = 0ull;
    LeafQueue leaves{L, lane};
    block_shares(on, b.x, b.y, b.z, b.c[0], b.c[1], b.c[2], leaves);
    leaves.sum(leaves.n);
    unsigned redo = 0u;
    if (!on) return redo;
    for_cells(b.c, ld.place(e, b.lo), [&](int i, int64_t at) {
        const double f = LaneShares::value(sum[i * kWaveTile]);
        if (f >= kSmallShare) ld.add(e, at, f);
        else if (fabs(f) >= kNoShare) redo |= 1u << i;
    });
    return redo;
}

// Recomputes one cell of a block alone (the paths first, first + stride, ... of exact_cell_share).  keep:
// this lane's LDS column.
template <class Loader>
__device__ __forceinline__ void clip_cell(const Loader& ld, int2 e, Block b, int cell, int first, int stride, double* keep) {
    const int q = int(udiv_small(unsigned(cell), unsigned(b.c[2]))), k = cell - q * b.c[2];
    const int a = int(udiv_small(unsigned(q), unsigned(b.c[1]))), j = q - a * b.c[1];
    for (int i = 0; i < 4; ++i) {
        b.x[i] -= double(a);
        b.y[i] -= double(j);
        b.z[i] -= double(k);
    }
    b.lo[0] += a;
    b.lo[1] += j;
    b.lo[2] += k;
    const double f = exact_cell_share(b.x, b.y, b.z, [&](int i) -> double& { return keep[i * kWaveTile]; }, first, stride);
    if (f > 0.0) ld.add(e, ld.place(e, b.lo).corner, f);
}

// A wavefront's state between calls of run_wave.
struct WaveState {
    unsigned pend = 0u;  // cells of this lane's last block left to the exact queue
    int2 pe = make_int2(0, 0);
    unsigned n_exact = 0, n_partial = 0;  // this lane's recomputes, the wave's clipped blocks
};

__device__ __forceinline__ void init_wave(BlockLds& L, int lane) {
    if (lane < 16) L.qn[lane] = 0;
    L.carry_key[lane] = -1;
    wave_sync();
}

// Feeds and clips until feed(L, lane) returns false (it appends at most one entry per lane), then, with
// `drain`, until the queues are empty: passes filled across the classes, a full queue or the exact one
// first.  Without `drain` every queue is left below 64 entries and nothing is carried.  A pass takes at
// least one entry and exact passes add none, so the loop ends.
template <class Feed, class Loader>
__device__ __forceinline__ void run_wave(BlockLds& L, int lane, WaveState& w, Feed& feed, const Loader& ld, bool drain) {
    bool draining = false;
    for (;;) {
        // pending cells go to the exact queue, one per lane and round, up to its 64 entries; a full exact
        // queue is clipped first
        const unsigned long long pm = __ballot(w.pend != 0u);
        const int nexact = pm ? __builtin_amdgcn_readfirstlane(L.qn[kExact]) : kWaveTile;
        if (nexact < kWaveTile) {
            const int room = kWaveTile - nexact;
            const int rank = mbcnt64(pm);
            if (w.pend && rank < room) {
                L.q[kExact][nexact + rank] = w.pe;
                L.cell[nexact + rank] = (unsigned char)__builtin_ctz(w.pend);
                w.pend &= w.pend - 1u;
                ++w.n_exact;
            }
            wave_sync();
            if (lane == 0) L.qn[kExact] = nexact + min(int(__popcll(pm)), room);
            wave_sync();
            continue;
        }
        // a queue to clip: full while there is work to feed, any non-empty one when draining
        const int qv = lane < kQueues ? L.qn[lane] : 0;
        const unsigned long long ready = __ballot(qv >= (draining ? 1 : kWaveTile));
        if (ready) {
            const int b = (ready >> kExact) & 1ull ? kExact : __builtin_ctzll(ready);
            const int cnt = __builtin_amdgcn_readfirstlane(__shfl(qv, b, 64));
            int2 e = make_int2(0, 0);
            int cell = 0, first = 0, stride = 1;
            bool have = false;
            if (draining && b != kExact && cnt < kWaveTile) {
                // up to 64 entries across all classes, from the top of each queue, lowest class first
                const int qc = lane < kClasses ? qv : 0;
                int pre = qc;
                for (int d = 1; d < 8; d <<= 1) {
                    const int o = __shfl_up(pre, d, 64);
                    if (lane >= d) pre += o;
                }
                const int excl = pre - qc;
                const int tq = lane < kClasses ? max(0, min(qc, kWaveTile - excl)) : 0;
                for (int qi = 0; qi < kClasses; ++qi) {
                    const int ex = __shfl(excl, qi, 64), tk = __shfl(tq, qi, 64), cq = __shfl(qc, qi, 64);
                    if (lane >= ex && lane < ex + tk) {
                        e = L.q[qi][cq - tk + (lane - ex)];
                        have = true;
                    }
                }
                wave_sync();
                if (lane < kClasses) L.qn[lane] = qc - tq;
            } else {
                // what the count holds beyond 64 are carried entries, which take the freed positions
                const int take = min(cnt, kWaveTile), rest = cnt - take;
                int at = lane;
                if (b == kExact && take <= kWaveTile / 4) {
                    // few cells (a drain): the lanes share each one's paths, or the wave would wait for the
                    // one with the most (196 608 tets on 64^3 cells: 424 us against 460)
                    const int bits = 31 - __builtin_clz(unsigned(kWaveTile / take));
                    const int shift = min(bits, 5);
                    stride = 1 << shift;
                    first = lane & (stride - 1);
                    at = lane >> shift;
                }
                if (at < take) {
                    e = L.q[b][at];
                    cell = L.cell[at];
                    have = true;
                }
                wave_sync();
                if (lane == 0) L.qn[b] = rest;
                if (rest > 0) {
                    const bool mine = L.carry_key[lane] == b;
                    const unsigned long long m = __ballot(mine);
                    if (mine) {
                        L.q[b][mbcnt64(m)] = L.carry[lane];
                        L.carry_key[lane] = -1;
                    }
                }
            }
            wave_sync();
            Block blk = {};
            if (have) blk = ld.block(e);
            if (b != kExact) {
                w.pend = clip_blocks(ld, have, e, blk, L, lane);
                w.pe = e;
            } else if (have) {
                clip_cell(ld, e, blk, cell, first, stride, &L.keep[0][lane]);
            }
            wave_sync();
            continue;
        }
        if (draining) break;
        if (!feed(L, lane)) {
            if (!drain) break;
            draining = true;
        }
    }
}

// Tile of 64 consecutive units over items of `cnt` units each (this lane's item: [start, start + cnt)):
// the item of unit `cursor + lane`, or -1 beyond the last.
__device__ __forceinline__ int item_of_unit(BlockLds& L, int lane, unsigned start, unsigned cnt, unsigned cursor) {
    L.mark[lane] = -1;
    wave_sync();
    if (cnt > 0 && start < cursor + kWaveTile && start + cnt > cursor) L.mark[int(max(start, cursor) - cursor)] = lane;
    wave_sync();
    int item = L.mark[lane];
    for (int d = 1; d < 64; d <<= 1) {
        const int o = __shfl_up(item, d, 64);
        if (lane >= d) item = max(item, o);
    }
    wave_sync();
    return item;
}

}  // namespace adeco
