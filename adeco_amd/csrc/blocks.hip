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
//                       the others go to one of 7 per-wave LDS queues by the number of x and y planes
//                       that cut the tet, so that the 64 lanes of a pass run through similar loops.  A
//                       full queue is clipped by the whole wave: each lane sums its block's shares in
//                       LDS (one column of kBlockCells doubles per lane) and adds tet_mass * share to
//                       the grid.  A share too small against the differences' rounding goes to one more
//                       queue whose passes recompute that cell alone from positive terms.
// Why blocks: the column form clips every column of a tet on its own, so a tet of 2 x 2 columns is cut by
// each inner plane twice over and through up to four nested stages of full 3-D pieces.  Here a plane is
// cut once for the cells on both its sides, a cut carries only the coordinates still needed and a
// piece's volume comes from edge ratios (4-5x fewer instructions per tet, 168 VGPRs: 3 waves per SIMD
// instead of 2).  256^3 clustered lattice, 16^3-cell leaves, 126 M pairs: 31.4 ms against 65.6 for the
// column form; 128^3: 3.8 against 7.1; 32^3-cell leaves on 97^3: 15.3 against 27.5.  It is also more
// accurate (128^3 leaf grids against 64-bit exact clipping: 9e-15 against 3e-13).  What bounds it:
// instruction issue at 40-50 % lane use, then FP64 atomics (one per cell a tet meets; the card takes
// 25-31 G/s of them scattered).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>

#include "../../include/adeco.h"
#include "batched_impl.hpp"
#include "block_clip.hpp"
#include "deposit_tet.hpp"
#include "kernels.hpp"
#include "runtime.hpp"
#include "wave_tiles.hpp"

namespace adeco {

namespace {

constexpr int kWaves = 4;  // wavefronts of a workgroup
constexpr int kThreads = 64 * kWaves;
constexpr int kClasses = 7;          // queues of blocks to clip
constexpr int kExact = kClasses;     // the queue of single cells to recompute
constexpr int kQueues = kClasses + 1;

// A queue entry: the pair, and the block's index in it with the source slot in the upper 6 bits (a
// pair has at most 512 * 512 * 256 = 2^26 blocks).
constexpr int kUnitBits = 26;
constexpr unsigned kUnitMask = (1u << kUnitBits) - 1u;

// Per-wavefront LDS.  An entry that finds its queue full is carried per lane and takes its place once
// that queue has been clipped; qn[b] counts queue b's entries and its carried ones.
struct BlockLds {
    int qn[16];
    int2 q[kQueues][kWaveTile];
    int2 carry[kWaveTile];
    signed char carry_key[kWaveTile];
    unsigned char cell[kWaveTile];  // of each exact-queue entry
    union {
        double acc[kBlockCells][kWaveTile];  // each lane's shares
        int mark[kWaveTile];                 // pair starts of the tile being classified
    };
};
// 3 workgroups of 4 waves share the 160 KB of a CU, which are handed out in pieces of 1280 bytes
static_assert((sizeof(BlockLds) * kWaves + 1279) / 1280 * 1280 * 3 <= 160 * 1024, "3 workgroups per CU");

// How a pair's covered cells are cut into blocks: blocks of b cells, n of them, per axis (x, y, z in
// the pair's order, extents ex <= ey <= ez).  z keeps up to 4 cells and x up to 2; the cells are
// spread evenly over an axis' blocks.  A pair of at most kBlockCells cells is one block.
struct BlockShape {
    int b[3], n[3];
};

__device__ __forceinline__ BlockShape block_shape(int ex, int ey, int ez) {
    BlockShape s;
    const bool one = ex * ey * ez <= kBlockCells;
    const int bz = one ? ez : min(ez, 4);
    const int bx = one ? ex : min(ex, 2);
    // cells left for y: 16 / (bx * bz), at least 2 (bx <= 2 and bz <= 4 unless `one`)
    const int room = one ? ey : (bx * bz <= 2 ? 8 : (bx * bz == 3 ? 5 : (bx * bz == 4 ? 4 : 2)));
    const int by = min(ey, room);
    const int e[3] = {ex, ey, ez}, b[3] = {bx, by, bz};
    for (int a = 0; a < 3; ++a) {
        const int n = b[a] >= e[a] ? 1 : int(udiv_small(unsigned(e[a] + b[a] - 1), unsigned(b[a])));
        s.b[a] = n == 1 ? e[a] : int(udiv_small(unsigned(e[a] + n - 1), unsigned(n)));
        s.n[a] = n == 1 ? 1 : int(udiv_small(unsigned(e[a] + s.b[a] - 1), unsigned(s.b[a])));
    }
    return s;
}

// Axis order of a pair, packed in 3 bits (PairData::range, bits 60-62): the axis of z and whether x and
// y are the next two axes in cyclic order or the reverse.
__device__ __forceinline__ int role_axis(int code, int role) {
    const int za = code & 3, u = za == 2 ? 0 : za + 1, v = u == 2 ? 0 : u + 1;
    const bool swap = code & 4;
    return role == 2 ? za : ((role == 0) != swap ? u : v);
}

template <class T>
__device__ __forceinline__ T pick(int a, T v0, T v1, T v2) {
    return a == 0 ? v0 : (a == 1 ? v1 : v2);
}

__global__ void __launch_bounds__(256) k_block_setup(LatticeView lat, PackedCorners ct, const int32_t* __restrict__ pairs,
                                                     int64_t n_pairs, const int64_t* __restrict__ n_dev,
                                                     const int64_t* __restrict__ grid_off, int n_grids,
                                                     const int32_t* __restrict__ pair_grid,
                                                     const GridDesc* __restrict__ grids, double tet_mass,
                                                     unsigned* __restrict__ cand, PairData* __restrict__ pd) {
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
        int lo[3], ext[3];
        for (int a = 0; a < 3; ++a) {
            const double c0 = comp(v[0], a), c1 = comp(v[1], a), c2 = comp(v[2], a), c3 = comp(v[3], a);
            const double mn = fmin(fmin(c0, c1), fmin(c2, c3)), mx = fmax(fmax(c0, c1), fmax(c2, c3));
            // the cells whose box can strictly overlap the tet's, widened by 1e-9 of a cell
            const int dm1 = g.dims - 1;
            int l = int(floor((mn - g.gmin[a]) / g.delta[a] - 1e-9));
            int h = int(floor((mx - g.gmin[a]) / g.delta[a] + 1e-9));
            l = l <= 0 ? 0 : (l >= dm1 ? dm1 : l);
            h = h <= 0 ? 0 : (h >= dm1 ? dm1 : h);
            lo[a] = l;
            ext[a] = h - l + 1;
        }
        const int za = ext[2] >= ext[1] && ext[2] >= ext[0] ? 2 : (ext[1] >= ext[0] ? 1 : 0);
        const int u = za == 2 ? 0 : za + 1, w = u == 2 ? 0 : u + 1;
        const bool swap = pick(w, ext[0], ext[1], ext[2]) < pick(u, ext[0], ext[1], ext[2]);
        const int code = za | (swap ? 4 : 0);
        const int ax = swap ? w : u, ay = swap ? u : w;
        const int ex = pick(ax, ext[0], ext[1], ext[2]), ey = pick(ay, ext[0], ext[1], ext[2]), ez = pick(za, ext[0], ext[1], ext[2]);
        const BlockShape s = block_shape(ex, ey, ez);
        const bool live = vol != 0.0;
        // positively oriented vertices in the pair's axis order (the face tests need the orientation)
        const bool flip = (vol < 0.0) != swap;
        unsigned long long* o = rows + threadIdx.x * (kWords + 1);
        for (int q = 0; q < 4; ++q) {
            const V3<double>& s0 = v[q];
            const int at = flip && (q == 0 || q == 3) ? 3 - q : q;
            const double c[3] = {g.scale[0] * (s0.x - g.gmin[0]), g.scale[1] * (s0.y - g.gmin[1]), g.scale[2] * (s0.z - g.gmin[2])};
            o[3 * at] = __double_as_longlong(pick(ax, c[0], c[1], c[2]));
            o[3 * at + 1] = __double_as_longlong(pick(ay, c[0], c[1], c[2]));
            o[3 * at + 2] = __double_as_longlong(pick(za, c[0], c[1], c[2]));
        }
        o[12] = __double_as_longlong(live ? tet_mass * (g.cell_vol / fabs(vol)) : 0.0);
        unsigned long long pack = (unsigned long long)code << 60;
        pack |= (unsigned long long)pick(ax, lo[0], lo[1], lo[2]) | (unsigned long long)ex << 30;
        pack |= (unsigned long long)pick(ay, lo[0], lo[1], lo[2]) << 10 | (unsigned long long)ey << 40;
        pack |= (unsigned long long)pick(za, lo[0], lo[1], lo[2]) << 20 | (unsigned long long)ez << 50;
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

// A block of a pair: its corner cell (pair's axis order), its sizes and the pair's vertices from the corner.
struct Block {
    int lo[3], c[3];
    double x[4], y[4], z[4];
};

__device__ __forceinline__ Block load_block(const PairData& pd, unsigned unit) {
    Block b;
    const unsigned long long rg = pd.range;
    const int ex = int(rg >> 30) & 1023, ey = int(rg >> 40) & 1023, ez = int(rg >> 50) & 1023;
    const BlockShape s = block_shape(ex, ey, ez);
    const unsigned rest = s.n[2] == 1 ? unit : udiv_small(unit, unsigned(s.n[2]));
    const int iz = int(unit - rest * unsigned(s.n[2]));
    const int ix = s.n[1] == 1 ? int(rest) : int(udiv_small(rest, unsigned(s.n[1])));
    const int iy = int(rest) - ix * s.n[1];
    b.lo[0] = int(rg & 1023u) + ix * s.b[0];
    b.lo[1] = int((rg >> 10) & 1023u) + iy * s.b[1];
    b.lo[2] = int((rg >> 20) & 1023u) + iz * s.b[2];
    b.c[0] = min(s.b[0], ex - ix * s.b[0]);
    b.c[1] = min(s.b[1], ey - iy * s.b[1]);
    b.c[2] = min(s.b[2], ez - iz * s.b[2]);
    for (int q = 0; q < 4; ++q) {
        b.x[q] = pd.S[3 * q] - double(b.lo[0]);
        b.y[q] = pd.S[3 * q + 1] - double(b.lo[1]);
        b.z[q] = pd.S[3 * q + 2] - double(b.lo[2]);
    }
    return b;
}

// Cell strides of the pair's axes in its grid.
struct Strides {
    int64_t x, y, z;
};
__device__ __forceinline__ Strides strides_of(unsigned long long range, int dims) {
    const int code = int(range >> 60) & 7;
    const int64_t s1 = dims, s2 = int64_t(dims) * dims;
    return Strides{pick(role_axis(code, 0), int64_t(1), s1, s2), pick(role_axis(code, 1), int64_t(1), s1, s2),
                   pick(role_axis(code, 2), int64_t(1), s1, s2)};
}

// Visits the cells of a block in the order of its shares: f(index, grid cell).
template <class F>
__device__ __forceinline__ void for_cells(const int c[3], int64_t corner, const Strides& st, F f) {
    const int n = c[0] * c[1] * c[2];
    int b = 0, k = 0;
    int64_t at = corner;
    const int64_t next_y = st.y - c[2] * st.z, next_x = st.x - c[1] * st.y;
    for (int i = 0; i < n; ++i) {
        f(i, at);
        at += st.z;
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

// Work class of a block to clip: by the planes that cut the tet across x and y (0, 1, more), and for a
// single x plane by whether it leaves one piece (1 or 3 vertices below) or three.  The class only
// groups blocks of similar loops.
__device__ __forceinline__ int work_class(const Block& b, const double mn[3], const double mx[3]) {
    const int fx = floor_clamped(mn[0], b.c[0]) + 1, lx = min(ceil_clamped(mx[0], b.c[0]) - 1, b.c[0]);
    const int fy = floor_clamped(mn[1], b.c[1]) + 1, ly = min(ceil_clamped(mx[1], b.c[1]) - 1, b.c[1]);
    const int px = lx - fx + 1, py = ly - fy + 1;
    if (px <= 0) return int(py >= 2);
    if (px >= 2) return 6;
    int n = 0;
    for (int q = 0; q < 4; ++q) n += int(b.x[q] < double(fx));
    return (py <= 1 ? 2 : 4) + int(n == 2);
}

// set bits of m below this lane
__device__ __forceinline__ int mbcnt64(unsigned long long m) {
    return int(__builtin_amdgcn_mbcnt_hi(unsigned(m >> 32), __builtin_amdgcn_mbcnt_lo(unsigned(m), 0u)));
}

// Classifies the 64 blocks of tile h.t of `src`: the filled ones are deposited, those to clip are
// appended to the wave's queues.
__device__ __forceinline__ void classify_tile(const TileSource& src, const TileHead& h, BlockLds& L, int lane,
                                              unsigned long long& n_partial) {
    const int np = h.np;
    const int64_t c0 = h.t * kWaveTile;
    L.mark[lane] = 0;
    wave_sync();
    // every pair owns >= 1 block, so pairs p0+1.. start at distinct positions 1..63
    if (lane >= 1 && lane < np && h.my_off - c0 < kWaveTile) L.mark[int(h.my_off - c0)] = lane;
    wave_sync();
    int in_tile = L.mark[lane];
    for (int d = 1; d < 64; d <<= 1) {
        const int o = __shfl_up(in_tile, d, 64);
        if (lane >= d) in_tile = max(in_tile, o);
    }
    const int64_t off = shfl_i64(h.my_off, in_tile);
    const int64_t c = c0 + lane;
    const int p = h.p0 + in_tile;
    const unsigned unit = unsigned(c - off);
    int key = -1;
    if (c < src.n_cand) {
        const PairData& pd = src.pd[p];
        if (pd.range) {
            const Block b = load_block(pd, unit);
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
            const bool single = b.c[0] * b.c[1] * b.c[2] == 1;
            if (hit) {
                int cls = CLS_PARTIAL;
                if (inside) {
                    if (single) cls = CLS_TET_IN_CELL;
                } else {
                    V3<double> s[4];
                    for (int q = 0; q < 4; ++q) s[q] = mk(b.x[q], b.y[q], b.z[q]);
                    cls = classify_margin(s, box);
                }
                if (cls == CLS_TET_IN_CELL || cls == CLS_CELL_IN_TET) {
                    const GridDesc& g = src.grids[pd.grid];
                    const Strides st = strides_of(pd.range, g.dims);
                    const int64_t corner = g.base + b.lo[0] * st.x + b.lo[1] * st.y + b.lo[2] * st.z;
                    const double m = cls == CLS_TET_IN_CELL ? src.tet_mass : pd.mcell;
                    for_cells(b.c, corner, st, [&](int, int64_t at) { unsafeAtomicAdd(src.grid_buf + at, m); });
                } else if (cls != CLS_NONE) {
                    key = work_class(b, mn, mx);
                }
            }
        }
    }
    // every queue holds < 64 entries here, so a count reaches at most 127; an entry beyond 64 is carried
    const int2 entry = make_int2(p, int(unit | unsigned(h.slot) << kUnitBits));
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
    n_partial += __popcll(__ballot(key >= 0));
    wave_sync();
}

// This lane's column of shares.
struct LaneShares {
    double* a;
    __device__ __forceinline__ void add(int i, double v) {
        __hip_atomic_fetch_add(a + i * kWaveTile, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    }
};

// Clips one queued block and deposits its cells, except those whose share is small against the
// rounding of the differences: returns their mask (bit = index of the cell in the block).
template <class Sources>
__device__ __forceinline__ unsigned clip_block(const Sources& srcs, int2 e, double* acc) {
    const TileSource& src = srcs.get(int(unsigned(e.y) >> kUnitBits));
    const PairData& pd = src.pd[e.x];
    const Block b = load_block(pd, unsigned(e.y) & kUnitMask);
    const int n = b.c[0] * b.c[1] * b.c[2];
    for (int i = 0; i < n; ++i) acc[i * kWaveTile] = 0.0;
    LaneShares sum{acc};
    block_shares(b.x, b.y, b.z, b.c[0], b.c[1], b.c[2], sum);
    const GridDesc& g = src.grids[pd.grid];
    const Strides st = strides_of(pd.range, g.dims);
    const int64_t corner = g.base + b.lo[0] * st.x + b.lo[1] * st.y + b.lo[2] * st.z;
    unsigned redo = 0u;
    for_cells(b.c, corner, st, [&](int i, int64_t at) {
        const double f = acc[i * kWaveTile];
        if (f >= kSmallShare) unsafeAtomicAdd(src.grid_buf + at, src.tet_mass * f);
        else if (fabs(f) >= kNoShare) redo |= 1u << i;
    });
    return redo;
}

// Recomputes one cell of a block alone.
template <class Sources>
__device__ __forceinline__ void clip_cell(const Sources& srcs, int2 e, int cell, double* keep) {
    const TileSource& src = srcs.get(int(unsigned(e.y) >> kUnitBits));
    const PairData& pd = src.pd[e.x];
    Block b = load_block(pd, unsigned(e.y) & kUnitMask);
    const int q = int(udiv_small(unsigned(cell), unsigned(b.c[2]))), k = cell - q * b.c[2];
    const int a = int(udiv_small(unsigned(q), unsigned(b.c[1]))), j = q - a * b.c[1];
    for (int i = 0; i < 4; ++i) {
        b.x[i] = pd.S[3 * i] - double(b.lo[0] + a);
        b.y[i] = pd.S[3 * i + 1] - double(b.lo[1] + j);
        b.z[i] = pd.S[3 * i + 2] - double(b.lo[2] + k);
    }
    const double f = exact_cell_share(b.x, b.y, b.z, [&](int i) -> double& { return keep[i * kWaveTile]; });
    const GridDesc& g = src.grids[pd.grid];
    const Strides st = strides_of(pd.range, g.dims);
    if (f > 0.0)
        unsafeAtomicAdd(src.grid_buf + g.base + (b.lo[0] + a) * st.x + (b.lo[1] + j) * st.y + (b.lo[2] + k) * st.z,
                        src.tet_mass * f);
}

// The persistent loop of one wavefront over work items [0, n_items): item -> (source slot, tile)
// directly or through `entries`.  The wave pops `chunk` items at a time; a queue reaching 64 entries is
// clipped at once; when the items run out the queues are drained, one pass per queue or (kMerge) in
// passes filled across the classes.  Every wave leaves once the counter passes n_items and its queues
// are empty: a pass takes at least one entry, and exact passes add none.
template <bool kMerge, class Sources>
__device__ __forceinline__ void wave_loop(const Sources& srcs, const int2* __restrict__ entries, int64_t n_items, int chunk,
                                          unsigned* __restrict__ queue_counter, unsigned long long* __restrict__ counters) {
    __shared__ BlockLds lds[kWaves];
    const int lane = threadIdx.x & 63;
    BlockLds& L = lds[threadIdx.x >> 6];
    if (lane < 16) L.qn[lane] = 0;
    L.carry_key[lane] = -1;
    wave_sync();
    unsigned long long n_partial = 0, n_exact = 0;
    int64_t it = 0, it_end = 0;
    TileHead head;  // of item `it` while it < it_end
    head.slot = head.p0 = head.np = 0;
    head.t = head.my_off = 0;
    bool draining = false;
    unsigned pend = 0u;  // cells of this lane's last block left to the exact queue
    int2 pe = make_int2(0, 0);
    for (;;) {
        // pending cells go to the exact queue, one per lane and round, up to its 64 entries; a full exact
        // queue is clipped first
        const unsigned long long pm = __ballot(pend != 0u);
        const int nexact = pm ? __builtin_amdgcn_readfirstlane(L.qn[kExact]) : kWaveTile;
        if (nexact < kWaveTile) {
            const int room = kWaveTile - nexact;
            const int rank = mbcnt64(pm);
            if (pend && rank < room) {
                L.q[kExact][nexact + rank] = pe;
                L.cell[nexact + rank] = (unsigned char)__builtin_ctz(pend);
                pend &= pend - 1u;
                ++n_exact;
            }
            wave_sync();
            if (lane == 0) L.qn[kExact] = nexact + min(int(__popcll(pm)), room);
            wave_sync();
            continue;
        }
        // a queue to clip: full while tiles remain, any non-empty one when draining; the exact queue first
        const int qv = lane < kQueues ? L.qn[lane] : 0;
        const unsigned long long ready = __ballot(qv >= (draining ? 1 : kWaveTile));
        if (ready) {
            const int b = (ready >> kExact) & 1ull ? kExact : __builtin_ctzll(ready);
            const int cnt = __builtin_amdgcn_readfirstlane(__shfl(qv, b, 64));
            int2 e = make_int2(0, 0);
            int cell = 0;
            bool have = false;
            if (kMerge && draining && b != kExact && cnt < kWaveTile) {
                // up to 64 entries across all classes, from the top of each queue, lowest class first
                const int qc = lane < kClasses ? qv : 0;
                int pre = qc;
                for (int d = 1; d < 16; d <<= 1) {
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
                if (lane < take) {
                    e = L.q[b][lane];
                    cell = L.cell[lane];
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
            if (b == kExact) {
                if (have) clip_cell(srcs, e, cell, &L.acc[0][lane]);
            } else if (have) {
                pend = clip_block(srcs, e, &L.acc[0][lane]);
                pe = e;
            }
            wave_sync();
            continue;
        }
        if (draining) break;
        if (it == it_end) {
            unsigned base = 0;
            if (lane == 0) base = atomicAdd(queue_counter, 1u);
            base = __builtin_amdgcn_readfirstlane(base);
            it = int64_t(base) * chunk;
            it_end = min(it + int64_t(chunk), n_items);
            if (it >= n_items) {
                draining = true;
                continue;
            }
            head = load_head(srcs, entries, it, lane);
        }
        const TileHead cur = head;
        ++it;
        if (it < it_end) head = load_head(srcs, entries, it, lane);
        classify_tile(srcs.get(cur.slot), cur, L, lane, n_partial);
    }
    if (lane == 0 && n_partial) atomicAdd(counters + 1, n_partial);
    if (n_exact) atomicAdd(counters, n_exact);
}

template <bool kMerge>
__global__ void __launch_bounds__(kThreads, 3) k_deposit_blocks(TileSource src, int chunk, unsigned* __restrict__ queue_counter,
                                                                unsigned long long* __restrict__ counters) {
    if (src.dev_sizes) {
        src.n_cand = src.dev_sizes[0];
        src.n_tiles = src.dev_sizes[1];
    }
    wave_loop<kMerge>(OneSource{src}, nullptr, src.n_tiles, chunk, queue_counter, counters);
}

template <bool kMerge>
__global__ void __launch_bounds__(kThreads, 3) k_step_blocks(const TileSource* __restrict__ sources,
                                                             const int2* __restrict__ entries, int n_entries, int chunk,
                                                             unsigned* __restrict__ queue_counter,
                                                             unsigned long long* __restrict__ counters) {
    wave_loop<kMerge>(ManySources{sources}, entries, n_entries, chunk, queue_counter, counters);
}

// This tet's shares on the host (the same code; tests only).
struct HostShares {
    double* a;
    void add(int i, double v) { a[i] += v; }
};

}  // namespace

hipError_t launch_block_setup(hipStream_t stream, const LatticeView& lat, const PackedCorners& ct, const int32_t* pairs,
                              int64_t n_pairs, const int64_t* n_dev, const int64_t* grid_off, int n_grids,
                              const int32_t* pair_grid, const GridDesc* d_grids, double tet_mass, unsigned* cand, PairData* pd) {
    hipLaunchKernelGGL(k_block_setup, dim3(unsigned((n_pairs + 255) / 256)), dim3(256), 0, stream, lat, ct, pairs, n_pairs,
                       n_dev, grid_off, n_grids, pair_grid, d_grids, tet_mass, cand, pd);
    return hipGetLastError();
}

int block_occupancy() {
    static std::atomic<int> cache;
    const int have = cache.load(std::memory_order_relaxed);
    if (have > 0) return have;
    int got = 0;
    const hipError_t e = hipOccupancyMaxActiveBlocksPerMultiprocessor(
        &got, reinterpret_cast<const void*>(k_deposit_blocks<false>), kThreads, 0);
    const int v = (e == hipSuccess && got > 0) ? got : 1;
    cache.store(v, std::memory_order_relaxed);  // concurrent first calls store the same value
    return v;
}

hipError_t launch_block_tiles(hipStream_t stream, const TileSource& src, unsigned* queue_counter,
                              unsigned long long* counters, int device) {
    const WaveLaunch w = wave_launch(src.n_tiles, block_occupancy(), kWaves, device);
    if (w.merge)
        hipLaunchKernelGGL(k_deposit_blocks<true>, dim3(w.grid), dim3(kThreads), 0, stream, src, w.chunk, queue_counter, counters);
    else
        hipLaunchKernelGGL(k_deposit_blocks<false>, dim3(w.grid), dim3(kThreads), 0, stream, src, w.chunk, queue_counter, counters);
    return hipGetLastError();
}

hipError_t launch_block_step(hipStream_t stream, const TileSource* d_sources, const int2* d_entries, int n_entries,
                             unsigned* queue_counter, unsigned long long* counters, int device) {
    const WaveLaunch w = wave_launch(n_entries, block_occupancy(), kWaves, device);
    if (w.merge)
        hipLaunchKernelGGL(k_step_blocks<true>, dim3(w.grid), dim3(kThreads), 0, stream, d_sources, d_entries, n_entries, w.chunk,
                           queue_counter, counters);
    else
        hipLaunchKernelGGL(k_step_blocks<false>, dim3(w.grid), dim3(kThreads), 0, stream, d_sources, d_entries, n_entries, w.chunk,
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
    for (int i = 0; i < n; ++i) shares[i] = 0.0;
    HostShares sum{shares};
    block_shares(x, y, z, cx, cy, cz, sum);
    for (int i = 0; i < n; ++i) {
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
