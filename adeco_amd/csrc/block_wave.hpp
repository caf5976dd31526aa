// Wavefront machinery of the block deposits (blocks.hip, direct.hip): the per-wave work queues, and the loop that
// clips what is in them.
//
// A block to clip is queued by its work class and a queue that holds 64 of them is clipped by the whole
// wave: each lane cuts its own block's tet, and the pieces (leaves) are gathered over the lanes and summed one
// per lane, each into its block's LDS column (LeafQueue).  A cell whose share is small against the rounding of
// the differences goes to one more queue, whose passes recompute it alone.
#pragma once

#include <hip/hip_runtime.h>

#include "batched_impl.hpp"
#include "block_cover.hpp"
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

// A lane's column of shares.
struct LaneShares {
    unsigned long long* a;
    __device__ __forceinline__ static long long term(double share) { return fixed_share(share); }
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
    const bool huge = b.full < kHugeTet;
    block_shares(on && !huge, b.x, b.y, b.z, b.c[0], b.c[1], b.c[2], leaves);
    leaves.sum(leaves.n);
    unsigned redo = 0u;
    if (!on) return redo;
    if (huge) return (1u << (b.c[0] * b.c[1] * b.c[2])) - 1u;
    const double small = small_share(b.y, b.z);
    for_cells(b.c, ld.place(e, b.lo), [&](int i, int64_t at) {
        const double f = from_fixed(sum[i * kWaveTile]);
        if (f >= small) ld.add(e, at, (fabs(f - b.full) <= kNearFull ? b.full : f) * b.scale);
        else if (fabs(f) >= kNoShare) redo |= 1u << i;
    });
    return redo;
}

// Recomputes one cell of a block alone (the paths first, first + stride, ... of exact_cell_share).  keep:
// this lane's LDS column.
template <class Loader>
__device__ __forceinline__ void clip_cell(const Loader& ld, int2 e, Block b, int cell, int first, int stride, double* keep) {
    b = cell_of(b, cell);
    const double f = exact_cell_share(b.x, b.y, b.z, [&](int i) -> double& { return keep[i * kWaveTile]; }, first, stride);
    if (f > 0.0) ld.add(e, ld.place(e, b.lo).corner, f * b.scale);
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
