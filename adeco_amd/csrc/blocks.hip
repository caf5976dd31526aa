// Batched persistent deposit over cell blocks: the FP64 form on grids of unit scaled cells.
//
// The unit of work (a candidate) is a block: up to kBlockCells cells of one (grid, tet) pair's
// covered range, cut and summed at once (block_clip.hpp).  Most tets of a leaf deposit are one block.
//   1. k_block_setup    one lane per pair: vertices scaled to cells in the pair's own axis order (z the
//                       longest covered extent, x the shortest), covered range, mass of a full cell ->
//                       one 128-byte PairData line and the number of blocks;
//   2. scan, tile map   as for the column form (batched.hip);
//   3. k_deposit_blocks persistent wavefronts pop chunks of tiles of 64 blocks.  Blocks that a face
//                       plane of the tet separates from it are dropped, blocks inside it are filled, and
//                       the others go to one of 8 per-wave LDS queues by the pieces that the x and y
//                       planes make, so that the 64 lanes of a pass run through similar loops.  A
//                       full queue is clipped by the whole wave: each lane cuts its block's tet, the
//                       pieces are summed one per lane into their blocks' LDS columns, and each lane adds
//                       tet_mass * share to the grid.  A share too small against the differences'
//                       rounding goes to one more queue whose passes recompute that cell alone from
//                       positive terms.
// Why blocks: the column form clips every column of a tet on its own, so a tet of 2 x 2 columns is cut by
// each inner plane twice over and through up to four nested stages of full 3-D pieces.  Here a plane is
// cut once for the cells on both its sides, a cut carries only the coordinates still needed and a
// piece's volume comes from edge ratios (4-5x fewer instructions per tet).  256^3 clustered lattice,
// 16^3-cell leaves, 126 M pairs: 31.6 ms against 65.6 for the column form; 128^3: 3.7 against 7.1;
// 32^3-cell leaves on 97^3: 15.3 against 27.5, and 9.6 with the pieces gathered over the lanes and blocks of
// 24 cells (block_wave.hpp).  It is also more accurate (128^3 leaf grids against 64-bit exact clipping:
// 5e-15 against 2e-13).  What bounds it: vector instructions (issued 80 % of the time with large tets, 52 %
// with small ones) at 65-75 % lane use, waiting at 2 waves per SIMD, and with small tets FP64 atomics (one per cell
// a tet meets: 17 % of the kernel, by a copy without them).  Two workgroups of 4 waves per CU: 20 KB of LDS a
// wave, and no spills (208 VGPRs; at 168 and 3 workgroups about 45 are spilled around each pass).
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

constexpr int kWaves = 4;  // wavefronts of a workgroup
constexpr int kThreads = 64 * kWaves;

// 2 workgroups of 4 waves share the 160 KB of a CU, which are handed out in pieces of 1280 bytes
static_assert((sizeof(BlockLds) * kWaves + 1279) / 1280 * 1280 * 2 <= 160 * 1024, "2 workgroups per CU");

// A queue entry: the pair, and the block's index in it with the source slot in the upper 6 bits.
constexpr int kUnitBits = 26;
static_assert(kMostBlocks <= 1u << kUnitBits, "bits of a block's index");
constexpr unsigned kUnitMask = (1u << kUnitBits) - 1u;

__global__ void __launch_bounds__(256) k_block_setup(LatticeView lat, PackedCorners ct, const int32_t* __restrict__ pairs,
                                                     int64_t n_pairs, const int64_t* __restrict__ n_dev,
                                                     const int64_t* __restrict__ grid_off, int n_grids,
                                                     const int32_t* __restrict__ pair_grid,
                                                     const GridDesc* __restrict__ grids, unsigned* __restrict__ cand,
                                                     PairData* __restrict__ pd) {
    // lines assembled in LDS rows of an odd number of words and stored as the block's contiguous,
    // non-temporal rows
    constexpr int kWords = int(sizeof(PairData) / 8);
    __shared__ unsigned long long rows[256 * (kWords + 1)];
    if (n_dev) n_pairs = min(*n_dev, n_pairs);
    const int64_t base = int64_t(blockIdx.x) * blockDim.x;
    if (base >= n_pairs) return;
    const int64_t p = base + threadIdx.x;
    if (p < n_pairs) {
        const int gi = pair_grid ? pair_grid[p] : (n_grids == 1 ? 0 : upper_bound_i64(grid_off, n_grids + 1, p) - 1);
        V3<double> v[4];
        lattice_tet_vertices(lat, ct, pairs[p], v);
        const GridDesc& g = grids[gi];
        const double vol = vol6(v[0], v[1], v[2], v[3]) / 6.0;
        TetCover t = cover_of(v, g);
        const BlockShape s = block_shape(t.e[0], t.e[1], t.e[2]);
        const bool live = has_volume(vol);
        orient(t, vol);
        unsigned long long* o = rows + threadIdx.x * (kWords + 1);
        for (int q = 0; q < 4; ++q)
            for (int r = 0; r < 3; ++r) o[3 * q + r] = __double_as_longlong(t.s[q][r]);
        o[12] = __double_as_longlong(live ? g.cell_vol / fabs(vol) : 0.0);
        unsigned long long pack = (unsigned long long)t.code << 60;
        for (int r = 0; r < 3; ++r) pack |= (unsigned long long)t.lo[r] << (10 * r) | (unsigned long long)t.e[r] << (30 + 10 * r);
        o[13] = live ? pack : 0ull;  // extent 0 marks a dead pair
        o[14] = (unsigned long long)unsigned(gi);
        o[15] = 0ull;
        cand[p] = live ? unsigned(s.n[0]) * unsigned(s.n[1]) * unsigned(s.n[2]) : 1u;
    }
    __syncthreads();
    const int rows_here = int(min(int64_t(256), n_pairs - base));
    unsigned long long* dst = reinterpret_cast<unsigned long long*>(pd + base);
    for (int k = threadIdx.x; k < rows_here * kWords; k += 256)
        __builtin_nontemporal_store(rows[(k / kWords) * (kWords + 1) + k % kWords], dst + k);
}

// The block of a queue entry from its pair's line, and the deposit of its shares.
template <class Sources>
struct PairLoader {
    const Sources& srcs;
    __device__ __forceinline__ static Block block_of(const PairData& pd, unsigned unit) {
        const unsigned long long rg = pd.range;
        const int lo[3] = {int(rg & 1023u), int((rg >> 10) & 1023u), int((rg >> 20) & 1023u)};
        const int e[3] = {int(rg >> 30) & 1023, int(rg >> 40) & 1023, int(rg >> 50) & 1023};
        double s[4][3];
        for (int q = 0; q < 4; ++q)
            for (int a = 0; a < 3; ++a) s[q][a] = pd.S[3 * q + a];
        return make_block(lo, e, s, pd.mcell, unit);
    }
    __device__ __forceinline__ Block block(int2 e) const {
        Block b = block_of(srcs.get(int(unsigned(e.y) >> kUnitBits)).pd[e.x], unsigned(e.y) & kUnitMask);
        shrink_tet(b);
        return b;
    }
    __device__ __forceinline__ Place place(int2 e, const int lo[3]) const {
        const TileSource& src = srcs.get(int(unsigned(e.y) >> kUnitBits));
        const PairData& pd = src.pd[e.x];
        const GridDesc& g = src.grids[pd.grid];
        Place p = place_of(lo, int(pd.range >> 60) & 7, g.dims);
        p.corner += g.base;
        return p;
    }
    __device__ __forceinline__ void add(int2 e, int64_t at, double share) const {
        const TileSource& src = srcs.get(int(unsigned(e.y) >> kUnitBits));
        unsafeAtomicAdd(src.grid_buf + at, src.tet_mass * share);
    }
};

// Feeds a wave from the work items [0, n_items): item -> (source slot, tile) directly or through
// `entries`, `chunk` items per access to the work queue.  Blocks inside the tet and tets inside a cell are
// deposited at once, empty blocks dropped.
template <class Sources>
struct TileFeed {
    const Sources& srcs;
    const int2* entries;
    int64_t n_items;
    int chunk;
    unsigned* queue_counter;
    WaveState& w;
    int64_t it = 0, it_end = 0;
    TileHead head;  // of item `it` while it < it_end

    __device__ __forceinline__ bool operator()(BlockLds& L, int lane) {
        if (it == it_end) {
            unsigned base = 0;
            if (lane == 0) base = atomicAdd(queue_counter, 1u);
            base = __builtin_amdgcn_readfirstlane(base);
            it = int64_t(base) * chunk;
            it_end = min(it + int64_t(chunk), n_items);
            if (it >= n_items) {
                it = it_end = n_items;
                return false;
            }
            head = load_head(srcs, entries, it, lane);
        }
        const TileHead h = head;
        ++it;
        if (it < it_end) head = load_head(srcs, entries, it, lane);
        const TileSource& src = srcs.get(h.slot);
        // every pair owns >= 1 block, so pairs p0+1.. start at distinct positions 1..63
        const int64_t c0 = h.t * kWaveTile;
        L.mark[lane] = 0;
        wave_sync();
        if (lane >= 1 && lane < h.np && h.my_off - c0 < kWaveTile) L.mark[int(h.my_off - c0)] = lane;
        wave_sync();
        int in_tile = L.mark[lane];
        for (int d = 1; d < 64; d <<= 1) {
            const int o = __shfl_up(in_tile, d, 64);
            if (lane >= d) in_tile = max(in_tile, o);
        }
        const int64_t off = shfl_i64(h.my_off, in_tile);
        const int p = h.p0 + in_tile;
        const unsigned unit = unsigned(c0 + lane - off);
        int key = kBlockEmpty;
        if (c0 + lane < src.n_cand) {
            const PairData& pd = src.pd[p];
            if (pd.range) {
                const Block b = PairLoader<Sources>::block_of(pd, unit);
                key = classify_block(b);
                if (key == kBlockTet || key == kBlockFull) {
                    const GridDesc& g = src.grids[pd.grid];
                    const double m = key == kBlockTet ? src.tet_mass : src.tet_mass * b.full;
                    double* grid = src.grid_buf + g.base;
                    for_cells(b.c, place_of(b.lo, int(pd.range >> 60) & 7, g.dims), [&](int, int64_t at) { unsafeAtomicAdd(grid + at, m); });
                }
            }
        }
        push_blocks(L, lane, key, make_int2(p, int(unit | unsigned(h.slot) << kUnitBits)));
        w.n_partial += unsigned(__popcll(__ballot(key >= 0)));
        return true;
    }
};

// The persistent loop of one wavefront.
template <class Sources>
__device__ __forceinline__ void deposit_tiles(const Sources& srcs, const int2* __restrict__ entries, int64_t n_items, int chunk,
                                              unsigned* __restrict__ queue_counter, unsigned long long* __restrict__ counters) {
    __shared__ BlockLds lds[kWaves];
    const int lane = threadIdx.x & 63;
    BlockLds& L = lds[threadIdx.x >> 6];
    init_wave(L, lane);
    WaveState w;
    TileFeed<Sources> feed{srcs, entries, n_items, chunk, queue_counter, w};
    feed.head.slot = feed.head.p0 = feed.head.np = 0;
    feed.head.t = feed.head.my_off = 0;
    run_wave(L, lane, w, feed, PairLoader<Sources>{srcs}, true);
    if (lane == 0 && w.n_partial) atomicAdd(counters + 1, (unsigned long long)w.n_partial);
    if (w.n_exact) atomicAdd(counters, (unsigned long long)w.n_exact);
}

__global__ void __launch_bounds__(kThreads, 2) k_deposit_blocks(TileSource src, int chunk, unsigned* __restrict__ queue_counter,
                                                                unsigned long long* __restrict__ counters) {
    if (src.dev_sizes) {
        src.n_cand = src.dev_sizes[0];
        src.n_tiles = src.dev_sizes[1];
    }
    deposit_tiles(OneSource{src}, nullptr, src.n_tiles, chunk, queue_counter, counters);
}

__global__ void __launch_bounds__(kThreads, 2) k_step_blocks(const TileSource* __restrict__ sources,
                                                             const int2* __restrict__ entries, int n_entries, int chunk,
                                                             unsigned* __restrict__ queue_counter,
                                                             unsigned long long* __restrict__ counters) {
    deposit_tiles(ManySources{sources}, entries, n_entries, chunk, queue_counter, counters);
}

// Shares summed on the host as the lanes of a wave do (the same code; tests only).
struct HostShares {
    unsigned long long* a;
    static long long term(double share) { return fixed_share(share); }
    void add(int i, long long v) { a[i] += (unsigned long long)v; }
};

}  // namespace

hipError_t launch_block_setup(hipStream_t stream, const LatticeView& lat, const PackedCorners& ct, const int32_t* pairs,
                              int64_t n_pairs, const int64_t* n_dev, const int64_t* grid_off, int n_grids,
                              const int32_t* pair_grid, const GridDesc* d_grids, unsigned* cand, PairData* pd) {
    hipLaunchKernelGGL(k_block_setup, dim3(unsigned((n_pairs + 255) / 256)), dim3(256), 0, stream, lat, ct, pairs, n_pairs,
                       n_dev, grid_off, n_grids, pair_grid, d_grids, cand, pd);
    return hipGetLastError();
}

int block_occupancy() {
    static std::atomic<int> cache;
    const int have = cache.load(std::memory_order_relaxed);
    if (have > 0) return have;
    int got = 0;
    const hipError_t e = hipOccupancyMaxActiveBlocksPerMultiprocessor(
        &got, reinterpret_cast<const void*>(k_deposit_blocks), kThreads, 0);
    const int v = (e == hipSuccess && got > 0) ? got : 1;
    cache.store(v, std::memory_order_relaxed);  // concurrent first calls store the same value
    return v;
}

hipError_t launch_block_tiles(hipStream_t stream, const TileSource& src, unsigned* queue_counter,
                              unsigned long long* counters, int device) {
    const WaveLaunch w = wave_launch(src.n_tiles, block_occupancy(), kWaves, device);
    hipLaunchKernelGGL(k_deposit_blocks, dim3(w.grid), dim3(kThreads), 0, stream, src, w.chunk, queue_counter, counters);
    return hipGetLastError();
}

hipError_t launch_block_step(hipStream_t stream, const TileSource* d_sources, const int2* d_entries, int n_entries,
                             unsigned* queue_counter, unsigned long long* counters, int device) {
    const WaveLaunch w = wave_launch(n_entries, block_occupancy(), kWaves, device);
    hipLaunchKernelGGL(k_step_blocks, dim3(w.grid), dim3(kThreads), 0, stream, d_sources, d_entries, n_entries, w.chunk,
                       queue_counter, counters);
    return hipGetLastError();
}

}  // namespace adeco

extern "C" int adeco_selftest_block_f64(const double* t, const int* cells3, double* shares, double* alone) {
    using namespace adeco;
    if (!t || !cells3 || !shares || !alone) return -1;
    const int cx = cells3[0], cy = cells3[1], cz = cells3[2], n = cx * cy * cz;
    if (cx < 1 || cy < 1 || cz < 1 || n > kBlockCells) return -1;
    double x[4], y[4], z[4];
    for (int q = 0; q < 4; ++q) {
        x[q] = t[3 * q];
        y[q] = t[3 * q + 1];
        z[q] = t[3 * q + 2];
    }
    unsigned long long sum[kBlockCells] = {};
    HostShares sums{sum};
    LeafSums<HostShares> leaves{sums};
    block_shares(true, x, y, z, cx, cy, cz, leaves);
    for (int i = 0; i < n; ++i) {
        shares[i] = from_fixed(sum[i]);
        const int k = i % cz, b = (i / cz) % cy, a = i / (cz * cy);
        double lx[4], ly[4], lz[4], keep[15];
        for (int q = 0; q < 4; ++q) {
            lx[q] = x[q] - a;
            ly[q] = y[q] - b;
            lz[q] = z[q] - k;
        }
        alone[i] = exact_cell_share(lx, ly, lz, [&](int j) -> double& { return keep[j]; });
    }
    return n;
}

// The block deposit of a tet soup on the host, block by block (the same code; tests only).
extern "C" int adeco_selftest_deposit_blocks_f64(const float* tets, int64_t n_tets, const float* bbox6, int dims, double tet_mass,
                                                 double* grid_out, int64_t* recomputes_out) {
    using namespace adeco;
    if (!tets || n_tets < 0 || !bbox6 || dims < 1 || dims > 1023 || !grid_out) return ADECO_EINVAL;
    const GridDesc g = make_grid_desc(make_grid_geom(bbox6, dims), 0);
    int64_t recomputes = 0;
    for (int64_t i = 0; i < n_tets; ++i) {
        V3<double> v[4];
        for (int q = 0; q < 4; ++q) v[q] = mk(double(tets[12 * i + 3 * q]), double(tets[12 * i + 3 * q + 1]), double(tets[12 * i + 3 * q + 2]));
        const double vol = vol6(v[0], v[1], v[2], v[3]);
        if (!has_volume(vol)) continue;
        TetCover t = cover_of(v, g);
        orient(t, vol);
        const double full = g.cell_vol / fabs(vol / 6.0);
        const BlockShape s = block_shape(t.e[0], t.e[1], t.e[2]);
        for (unsigned u = 0; u < unsigned(s.n[0] * s.n[1] * s.n[2]); ++u) {
            Block b = make_block(t.lo, t.e, t.s, full, u);
            const int key = classify_block(b);
            if (key == kBlockEmpty) continue;
            const Place p = place_of(b.lo, t.code, dims);
            if (key < 0) {
                const double m = key == kBlockTet ? tet_mass : tet_mass * full;
                for_cells(b.c, p, [&](int, int64_t at) { grid_out[at] += m; });
                continue;
            }
            shrink_tet(b);
            unsigned long long sum[kBlockCells] = {};
            HostShares shares{sum};
            LeafSums<HostShares> leaves{shares};
            const bool huge = b.full < kHugeTet;
            block_shares(!huge, b.x, b.y, b.z, b.c[0], b.c[1], b.c[2], leaves);
            const double small = small_share(b.y, b.z);
            for_cells(b.c, p, [&](int c, int64_t at) {
                double f = from_fixed(sum[c]), keep[15];
                if (fabs(f - b.full) <= kNearFull) f = b.full;
                if (f < small || huge) {
                    if (fabs(f) < kNoShare && !huge) return;
                    const Block cell = cell_of(b, c);
                    f = exact_cell_share(cell.x, cell.y, cell.z, [&](int j) -> double& { return keep[j]; });
                    ++recomputes;
                }
                if (f > 0.0) grid_out[at] += tet_mass * f * b.scale;
            });
        }
    }
    if (recomputes_out) *recomputes_out = recomputes;
    return ADECO_OK;
}
