// Direct block deposit: tets straight from their vertices onto their grids in a single launch, with no pair
// lines, scan or tile map in between (the FP64 deposit on grids of unit scaled cells: the plain forms, and
// the leaf deposit where most pairs are a block or two).
//
// A wavefront takes `per_item` consecutive tets from a work counter, one per lane: covered range and
// number of blocks (block_wave.hpp).  The blocks of the item are then walked 64 at a time, one per lane;
// each lane reads its block's vertices again (they are in cache), classifies the block and queues it,
// and full queues are clipped by the whole wave.  So a wave's lanes share the cells of a large tet, and
// nothing but the tets is read from memory.
// Against the one-tet-per-thread kernel (deposit.hip), whose waves run as long as their largest tet
// walks its cells: one meta-patch of 2 058 tets on 16^3 cells 37 us against 900-1130, a leaf's 98 784 tets
// on 16^3 cells 115 against 1420-1530, 196 608 tets on 64^3 cells 0.28 ms against 3.8.  All leaves of an
// octree in one launch instead of one each: 64 leaves, 1.86 M pairs, 16^3 cells 0.66 ms against 15.2.
// What bounds it: a small launch lasts as long as one wave's chain of passes (classify, clip, recompute:
// 20-30 us each, at mostly one wave per SIMD); a large one is bound as the batched form is (blocks.hip).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>

#include "../../include/adeco.h"
#include "batched_impl.hpp"
#include "block_wave.hpp"
#include "deposit_tet.hpp"
#include "kernels.hpp"
#include "runtime.hpp"

namespace adeco {

namespace {

constexpr int kWaves = 4;
constexpr int kThreads = 64 * kWaves;
static_assert((sizeof(BlockLds) * kWaves + 1279) / 1280 * 1280 * 2 <= 160 * 1024, "2 workgroups per CU");

// Tets of one grid.
struct OneGrid {
    GridDesc g;
    __device__ __forceinline__ const GridDesc& grid(int) const { return g; }
};

// The tets of a lattice: all of them, or those listed.
struct LatticeTets : OneGrid {
    LatticeView lat;
    PackedCorners ct;
    const int32_t* ids;
    __device__ __forceinline__ bool fetch(int64_t i, V3<double> v[4]) const {
        lattice_tet_vertices(lat, ct, ids ? int64_t(ids[i]) : i, v);
        return true;
    }
};

// The (leaf, tet) pairs of an octree, each with the grid of its leaf.
struct LeafTets {
    LatticeView lat;
    PackedCorners ct;
    const int32_t* pairs;
    const int32_t* pair_grid;
    const GridDesc* grids;
    __device__ __forceinline__ const GridDesc& grid(int i) const { return grids[pair_grid[i]]; }
    __device__ __forceinline__ bool fetch(int64_t i, V3<double> v[4]) const {
        lattice_tet_vertices(lat, ct, pairs[i], v);
        return true;
    }
};

// A tet soup: 4 vertices of 3 floats each.
struct SoupTets : OneGrid {
    const float* p;
    __device__ __forceinline__ bool fetch(int64_t i, V3<double> v[4]) const {
        const float* t = p + 12 * i;
        for (int q = 0; q < 4; ++q) v[q] = mk(double(t[3 * q]), double(t[3 * q + 1]), double(t[3 * q + 2]));
        return true;
    }
};

// The 6 tets of every cell of meta-patches of m^3 cells (AoS positions); a cell with a 666 sentinel
// vertex has none (AdDepositTets2Grid.h:1029-1038).
struct PatchTets : OneGrid {
    const float* pos;
    int m;
    PackedCorners pc;
    __device__ __forceinline__ bool fetch(int64_t i, V3<double> v[4]) const {
        const unsigned cell = unsigned(i / 6), cpp = unsigned(m * m * m);
        const int lt = int(i - int64_t(cell) * 6);
        const unsigned p = cell / cpp, c = cell - p * cpp, mm = unsigned(m * m);
        const unsigned ck = c / mm, rest = c - ck * mm, cj = rest / unsigned(m), ci = rest - cj * unsigned(m);
        const int ay = 3 * (m + 1), az = ay * (m + 1);
        const float* base = pos + int64_t(p) * az * (m + 1) + 3 * int(ci) + ay * int(cj) + az * int(ck);
        bool whole = true;
        for (int s = 0; s < 8; ++s) {
            const float* q = base + 3 * (s & 1) + ay * ((s >> 1) & 1) + az * (s >> 2);
            whole = whole && !is_sentinel(q[0], q[1], q[2]);
        }
        for (int q = 0; q < 4; ++q) {
            const int code = pc.code(lt, q);
            const float* pv = base + 3 * (code & 1) + ay * ((code >> 1) & 1) + az * ((code >> 2) & 1);
            v[q] = mk(double(pv[0]), double(pv[1]), double(pv[2]));
        }
        return whole;
    }
};

// An entry is the tet's index in the launch and the block's index in the tet.
template <class Tets>
struct DirectLoader {
    const Tets& tets;
    double* grid;
    double tet_mass;
    __device__ __forceinline__ Block block(int2 e) const {
        V3<double> v[4];
        (void)tets.fetch(e.x, v);
        const GridDesc& g = tets.grid(e.x);
        TetCover t = cover_of(v, g);
        const double vol = vol6(v[0], v[1], v[2], v[3]);
        orient(t, vol);
        Block b = make_block(t.lo, t.e, t.s, qdiv(6.0 * g.cell_vol, fabs(vol)), unsigned(e.y) & kUnits);
        shrink_tet(b);
        return b;
    }
    __device__ __forceinline__ Place place(int2 e, const int lo[3]) const {
        const GridDesc& g = tets.grid(e.x);
        Place p = place_of(lo, int(unsigned(e.y) >> 29), g.dims);
        p.corner += g.base;
        return p;
    }
    __device__ __forceinline__ void add(int2, int64_t at, double share) const { unsafeAtomicAdd(grid + at, tet_mass * share); }
    static constexpr unsigned kUnits = (1u << 29) - 1u;  // below the axis order's 3 bits
};

template <class Tets>
struct DirectFeed {
    const Tets& tets;
    double* grid;
    double tet_mass;
    unsigned n_tets, per_item, per_pop;
    unsigned* counter;
    WaveState& w;
    int64_t n_units = 0;
    // the tets taken from the counter and not yet begun; the current item: its first tet, this lane's blocks
    // [start, start + cnt), their total, and the next block to walk
    unsigned next = 0, end = 0, first = 0;
    unsigned start = 0, cnt = 0, total = 0, cursor = 0;

    // One step: a new item (whose blocks follow at once when no tet has more than one), or the next 64
    // blocks of the current one.
    __device__ __forceinline__ bool operator()(BlockLds& L, int lane) {
        const bool fresh = cursor >= total;
        unsigned t;  // this lane's tet, its block below
        bool live;
        unsigned unit = 0;
        if (fresh) {
            if (next >= end) {
                unsigned pop = 0;
                if (lane == 0) pop = atomicAdd(counter, 1u);
                const int64_t at = int64_t(__builtin_amdgcn_readfirstlane(pop)) * per_pop;
                if (at >= n_tets) return false;
                next = unsigned(at);
                end = unsigned(min(at + per_pop, int64_t(n_tets)));
            }
            first = next;
            next += per_item;
            t = first + unsigned(lane);
            live = unsigned(lane) < per_item && t < end;
            n_units += __popcll(__ballot(live));  // (a tet that deposits nothing counts as one block)
        } else {
            const int item = item_of_unit(L, lane, start, cnt, cursor);
            const unsigned item_start = unsigned(__shfl(int(start), max(item, 0), 64));
            t = first + unsigned(max(item, 0));
            live = cursor + unsigned(lane) < total;
            unit = cursor + unsigned(lane) - item_start;
            cursor += kWaveTile;
        }
        int key = kBlockEmpty, code = 0;
        double vol = 0.0;
        TetCover c;
        if (live) {
            V3<double> v[4];
            live = tets.fetch(t, v);
            c = cover_of(v, tets.grid(int(t)));
            code = c.code;
            vol = vol6(v[0], v[1], v[2], v[3]);
            live = live && has_volume(vol);
        }
        if (fresh) {
            cnt = 0;
            if (live) {
                const BlockShape s = block_shape(c.e[0], c.e[1], c.e[2]);
                cnt = unsigned(s.n[0]) * unsigned(s.n[1]) * unsigned(s.n[2]);
            }
            cursor = total = 0;
            if (__ballot(cnt > 1)) {
                unsigned last = cnt;
                for (int d = 1; d < 64; d <<= 1) {
                    const unsigned o = unsigned(__shfl_up(int(last), d, 64));
                    if (lane >= d) last += o;
                }
                start = last - cnt;
                total = unsigned(__builtin_amdgcn_readlane(int(last), 63));
                n_units += int64_t(total) - __popcll(__ballot(cnt > 0));
                return true;
            }
        }
        if (live) {
            orient(c, vol);
            const Block b = make_block(c.lo, c.e, c.s, 1.0, unit);
            key = classify_block(b);
            if (key == kBlockTet || key == kBlockFull) {
                const GridDesc& g = tets.grid(int(t));
                const double m = key == kBlockTet ? tet_mass : tet_mass * (g.cell_vol / fabs(vol / 6.0));
                double* to = grid + g.base;
                for_cells(b.c, place_of(b.lo, code, g.dims), [&](int, int64_t at) { unsafeAtomicAdd(to + at, m); });
            }
        }
        push_blocks(L, lane, key, make_int2(int(t), int(unit | unsigned(code) << 29)));
        w.n_partial += unsigned(__popcll(__ballot(key >= 0)));
        return true;
    }
};

template <class Tets>
__global__ void __launch_bounds__(kThreads, 2) k_deposit_direct(Tets tets, unsigned n_tets, unsigned per_item, unsigned per_pop,
                                                                double tet_mass, double* __restrict__ grid,
                                                                DirectCounters* __restrict__ ctr) {
    __shared__ BlockLds lds[kWaves];
    const int lane = threadIdx.x & 63;
    BlockLds& L = lds[threadIdx.x >> 6];
    init_wave(L, lane);
    WaveState w;
    DirectFeed<Tets> feed{tets, grid, tet_mass, n_tets, per_item, per_pop, &ctr->next, w};
    run_wave(L, lane, w, feed, DirectLoader<Tets>{tets, grid, tet_mass}, true);
    if (lane == 0 && w.n_partial) atomicAdd(&ctr->partials, (unsigned long long)w.n_partial);
    if (lane == 0 && feed.n_units) atomicAdd(&ctr->units, (unsigned long long)feed.n_units);
    if (w.n_exact) atomicAdd(&ctr->recomputes, (unsigned long long)w.n_exact);
}

template <class Tets>
hipError_t launch(const Tets& tets, int64_t n_tets, bool small_tets, double tet_mass, double* grid, DirectCounters* ctr,
                  int device, hipStream_t stream) {
    if (n_tets <= 0) return hipSuccess;
    int cus = 256;
    (void)hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, device);
    // tets per item: 64 fill a wave's lanes; fewer where that leaves 7 of 8 resident waves without work.  (A small
    // launch is over when its slowest wave is, so a wave's chain of passes should be short; but passes with
    // few lanes cost as much as full ones and get in each other's way.  2 058 tets on 16^3 cells, the call: two
    // items per resident wave 160 us, one for half 120, for a quarter or an eighth 90-100; 98 784 tets: 343, 285,
    // 282 us; 196 608 tets on 64^3 cells: 457, 445, 440.)
    const int64_t waves = int64_t(cus) * 2 * kWaves;
    static_assert(64ull * kMostBlocks + kWaveTile < 1ull << 32, "the blocks of an item's tets are counted in 32 bits");
    int per_item = kWaveTile;
    while (per_item > 1 && 8 * n_tets < waves * per_item) per_item >>= 1;
    const int64_t items = (n_tets + per_item - 1) / per_item;
    const WaveLaunch w = wave_launch(items, block_occupancy(), kWaves, device);
    // items per pop: one where the tets' blocks may differ much in number (45 M blocks of 6.7 M pairs on 32^3-cell
    // leaves: 18.3 ms against 23.2 with 4), else up to the launch shape's with at least 8 pops per wave (15.3 M
    // pairs on 16^3-cell leaves: 4.19 ms against 4.37 with 1)
    const int64_t chunk = small_tets ? std::max<int64_t>(1, std::min<int64_t>(w.chunk, items / (8 * waves))) : 1;
    hipLaunchKernelGGL(k_deposit_direct<Tets>, dim3(w.grid), dim3(kThreads), 0, stream, tets, unsigned(n_tets), unsigned(per_item),
                       unsigned(per_item * chunk), tet_mass, grid, ctr);
    return hipGetLastError();
}

}  // namespace

bool direct_deposit_fits(const GridDesc* grids, int64_t n, int64_t n_tets) {
    // unit scaled cells (block planes are shared by neighbouring cells), block indices of 29 bits and tet
    // indices of 31
    return deposit_form(ADECO_PREC_FP64, grids, n) == kFormBlocks && grids[0].dims <= 1023 && n_tets < (int64_t(1) << 31) - 2;
}

bool direct_deposit_fits(const GridGeom& g, int64_t n_tets) {
    const GridDesc d = make_grid_desc(g, 0);
    return direct_deposit_fits(&d, 1, n_tets);
}

hipError_t launch_direct_lattice(const LatticeView& lat, int decomp, const int32_t* d_ids, int64_t n_tets, const GridGeom& g,
                                 double tet_mass, double* d_grid, DirectCounters* ctr, int device, hipStream_t stream) {
    return launch(LatticeTets{{make_grid_desc(g, 0)}, lat, pack_corners(corner_table(decomp)), d_ids}, n_tets, false, tet_mass,
                  d_grid, ctr, device, stream);
}

hipError_t launch_direct_leaves(const LatticeView& lat, int decomp, const int32_t* d_pairs, const int32_t* d_pair_grid,
                                int64_t n_pairs, const GridDesc* d_grids, bool small_tets, double tet_mass,
                                double* d_grid_buf, DirectCounters* ctr, int device, hipStream_t stream) {
    return launch(LeafTets{lat, pack_corners(corner_table(decomp)), d_pairs, d_pair_grid, d_grids}, n_pairs, small_tets, tet_mass,
                  d_grid_buf, ctr, device, stream);
}

hipError_t launch_direct_soup(const float* d_tets, int64_t n_tets, const GridGeom& g, double tet_mass, double* d_grid,
                              DirectCounters* ctr, int device, hipStream_t stream) {
    return launch(SoupTets{{make_grid_desc(g, 0)}, d_tets}, n_tets, false, tet_mass, d_grid, ctr, device, stream);
}

hipError_t launch_direct_patches(const float* d_pos, int64_t num_patches, int m, int decomp, const GridGeom& g, double tet_mass,
                                 double* d_grid, DirectCounters* ctr, int device, hipStream_t stream) {
    return launch(PatchTets{{make_grid_desc(g, 0)}, d_pos, m, pack_corners(corner_table(decomp))}, num_patches * m * m * m * 6,
                  false, tet_mass, d_grid, ctr, device, stream);
}

}  // namespace adeco
