// Direct block deposit: tets straight from their vertices onto one grid in a single launch, with no pair
// lines, scan or tile map in between (the plain form of the FP64 deposit on grids of unit scaled cells).
//
// A wavefront takes `per_item` consecutive tets from a work counter, one per lane: covered range and
// number of blocks (block_wave.hpp).  The blocks of the item are then walked 64 at a time, one per lane;
// each lane reads its block's vertices again (they are in cache), classifies the block and queues it,
// and full queues are clipped by the whole wave.  So a wave's lanes share the cells of a large tet, and
// nothing but the tets is read from memory.
// Against the one-tet-per-thread kernel (deposit.hip), whose waves run as long as their largest tet
// walks its cells: one meta-patch of 2 058 tets on 16^3 cells 110 us against 900-1130, a leaf's 98 784 tets
// on 16^3 cells 205 against 1420-1530, 196 608 tets on 64^3 cells 0.42 ms against 3.8.  What bounds it: a
// small launch lasts as long as one wave's chain of passes (classify, clip, recompute: 20-30 us each, at
// mostly one wave per SIMD); a large one is bound as the batched form is (blocks.hip).
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
constexpr int kCells = 16;
using Lds = BlockLds<kCells>;
static_assert((sizeof(Lds) * kWaves + 1279) / 1280 * 1280 * 3 <= 160 * 1024, "3 workgroups per CU");

// The tets of a lattice: all of them, or those listed.
struct LatticeTets {
    LatticeView lat;
    PackedCorners ct;
    const int32_t* ids;
    __device__ __forceinline__ bool fetch(int64_t i, V3<double> v[4]) const {
        lattice_tet_vertices(lat, ct, ids ? int64_t(ids[i]) : i, v);
        return true;
    }
};

// A tet soup: 4 vertices of 3 floats each.
struct SoupTets {
    const float* p;
    __device__ __forceinline__ bool fetch(int64_t i, V3<double> v[4]) const {
        const float* t = p + 12 * i;
        for (int q = 0; q < 4; ++q) v[q] = mk(double(t[3 * q]), double(t[3 * q + 1]), double(t[3 * q + 2]));
        return true;
    }
};

// The 6 tets of every cell of meta-patches of m^3 cells (AoS positions); a cell with a 666 sentinel
// vertex has none (AdDepositTets2Grid.h:1029-1038).
struct PatchTets {
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

// A tet in the cells of a grid: its cover and its vertices, in the cover's axis order.
struct TetCover {
    int lo[3], e[3], code;
    double s[4][3];
};

__device__ __forceinline__ TetCover cover_of(const V3<double> v[4], const GridDesc& g) {
    double c[4][3];
    int lo[3], e[3];
    for (int a = 0; a < 3; ++a) {
        for (int q = 0; q < 4; ++q) c[q][a] = g.scale[a] * (comp(v[q], a) - g.gmin[a]);
        int h;
        covered(fmin(fmin(c[0][a], c[1][a]), fmin(c[2][a], c[3][a])), fmax(fmax(c[0][a], c[1][a]), fmax(c[2][a], c[3][a])), g.dims,
                lo[a], h);
        e[a] = h - lo[a] + 1;
    }
    TetCover t;
    t.code = role_code(e);
    for (int r = 0; r < 3; ++r) {
        const int a = role_axis(t.code, r);
        t.lo[r] = pick(a, lo[0], lo[1], lo[2]);
        t.e[r] = pick(a, e[0], e[1], e[2]);
        for (int q = 0; q < 4; ++q) t.s[q][r] = pick(a, c[q][0], c[q][1], c[q][2]);
    }
    return t;
}

// An entry is the tet's index in the launch and the block's index in the tet.
template <class Tets>
struct DirectLoader {
    const Tets& tets;
    const GridDesc& g;
    double* grid;
    double tet_mass;
    __device__ __forceinline__ Block block(int2 e) const {
        V3<double> v[4];
        (void)tets.fetch(e.x, v);
        const TetCover t = cover_of(v, g);
        return make_block<kCells>(t.lo, t.e, t.s, unsigned(e.y) & kUnits);
    }
    __device__ __forceinline__ Place place(int2 e, const int lo[3]) const { return place_of(lo, int(unsigned(e.y) >> 29), g.dims); }
    __device__ __forceinline__ void add(int2, int64_t at, double share) const { unsafeAtomicAdd(grid + at, tet_mass * share); }
    static constexpr unsigned kUnits = (1u << 29) - 1u;  // below the axis order's 3 bits
};

template <class Tets>
struct DirectFeed {
    const Tets& tets;
    const GridDesc& g;
    double* grid;
    double tet_mass;
    int64_t n_tets;
    int per_item;
    unsigned* counter;
    WaveState& w;
    int64_t n_units = 0;
    // the current item: its first tet, this lane's blocks [start, start + cnt), their total, and the next
    // block to walk
    int64_t first = 0;
    unsigned start = 0, cnt = 0, total = 0, cursor = 0;

    // One step: a new item (whose blocks follow at once when no tet has more than one), or the next 64
    // blocks of the current one.
    __device__ __forceinline__ bool operator()(Lds& L, int lane) {
        const bool fresh = cursor >= total;
        int64_t t;  // this lane's tet, its block below
        bool live;
        unsigned unit = 0;
        if (fresh) {
            unsigned item = 0;
            if (lane == 0) item = atomicAdd(counter, 1u);
            first = int64_t(__builtin_amdgcn_readfirstlane(item)) * per_item;
            if (first >= n_tets) return false;
            t = first + lane;
            live = lane < per_item && t < n_tets;
        } else {
            const int item = item_of_unit(L, lane, start, cnt, cursor);
            const unsigned item_start = unsigned(__shfl(int(start), max(item, 0), 64));
            t = first + item;
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
            c = cover_of(v, g);
            code = c.code;
            vol = vol6(v[0], v[1], v[2], v[3]);
            live = live && vol != 0.0;
        }
        if (fresh) {
            cnt = 0;
            if (live) {
                const BlockShape s = block_shape<kCells>(c.e[0], c.e[1], c.e[2]);
                cnt = unsigned(s.n[0]) * unsigned(s.n[1]) * unsigned(s.n[2]);
            }
            cursor = total = 0;
            if (__ballot(cnt > 1)) {
                unsigned end = cnt;
                for (int d = 1; d < 64; d <<= 1) {
                    const unsigned o = unsigned(__shfl_up(int(end), d, 64));
                    if (lane >= d) end += o;
                }
                start = end - cnt;
                total = unsigned(__builtin_amdgcn_readlane(int(end), 63));
                n_units += total;
                return true;
            }
            n_units += __popcll(__ballot(live));
        }
        if (live) {
            // positively oriented in the cover's axis order (the face tests need it)
            if ((vol < 0.0) != bool(code & 4))
                for (int a = 0; a < 3; ++a) {
                    const double s0 = c.s[0][a];
                    c.s[0][a] = c.s[3][a];
                    c.s[3][a] = s0;
                }
            const Block b = make_block<kCells>(c.lo, c.e, c.s, unit);
            key = classify_block(b);
            if (key == kBlockTet || key == kBlockFull) {
                const double m = key == kBlockTet ? tet_mass : tet_mass * (g.cell_vol / fabs(vol / 6.0));
                for_cells(b.c, place_of(b.lo, code, g.dims), [&](int, int64_t at) { unsafeAtomicAdd(grid + at, m); });
            }
        }
        push_blocks(L, lane, key, make_int2(int(t), int(unit | unsigned(code) << 29)));
        w.n_partial += unsigned(__popcll(__ballot(key >= 0)));
        return true;
    }
};

template <class Tets>
__global__ void __launch_bounds__(kThreads, 3) k_deposit_direct(Tets tets, int64_t n_tets, int per_item, GridDesc g, double tet_mass,
                                                                double* __restrict__ grid, DirectCounters* __restrict__ ctr) {
    __shared__ Lds lds[kWaves];
    const int lane = threadIdx.x & 63;
    Lds& L = lds[threadIdx.x >> 6];
    init_wave(L, lane);
    WaveState w;
    DirectFeed<Tets> feed{tets, g, grid, tet_mass, n_tets, per_item, &ctr->next, w};
    run_wave(L, lane, w, feed, DirectLoader<Tets>{tets, g, grid, tet_mass}, true);
    if (lane == 0 && w.n_partial) atomicAdd(&ctr->partials, (unsigned long long)w.n_partial);
    if (lane == 0 && feed.n_units) atomicAdd(&ctr->units, (unsigned long long)feed.n_units);
    if (w.n_exact) atomicAdd(&ctr->recomputes, (unsigned long long)w.n_exact);
}

template <class Tets>
hipError_t launch(const Tets& tets, int64_t n_tets, const GridDesc& g, double tet_mass, double* grid, DirectCounters* ctr,
                  int device, hipStream_t stream) {
    if (n_tets <= 0) return hipSuccess;
    int cus = 256;
    (void)hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, device);
    // tets per item: 64 fill a wave's lanes; fewer where that leaves resident waves without work (a small
    // launch is over when its slowest wave is, and large tets bring many blocks each): about two items
    // per resident wave
    const int64_t waves = int64_t(cus) * 3 * kWaves;
    // (64 tets of up to 2^26 blocks each would overflow their 32-bit sum on grids beyond 512^3)
    int per_item = g.dims <= 512 ? 64 : 32;
    while (per_item > 1 && n_tets < 2 * waves * per_item) per_item >>= 1;
    const int64_t items = (n_tets + per_item - 1) / per_item;
    const unsigned blocks = unsigned(std::min<int64_t>((items + kWaves - 1) / kWaves, int64_t(cus) * 3));
    hipLaunchKernelGGL(k_deposit_direct<Tets>, dim3(blocks), dim3(kThreads), 0, stream, tets, n_tets, per_item, g, tet_mass, grid,
                       ctr);
    return hipGetLastError();
}

}  // namespace

bool direct_deposit_fits(const GridGeom& g, int64_t n_tets) {
    // unit scaled cells (block planes are shared by neighbouring cells), block indices of 29 bits and tet
    // indices of 31
    const GridDesc d = make_grid_desc(g, 0);
    return deposit_form(ADECO_PREC_FP64, &d, 1) == kFormBlocks && g.dims <= 1023 && n_tets < (int64_t(1) << 31);
}

hipError_t launch_direct_lattice(const LatticeView& lat, int decomp, const int32_t* d_ids, int64_t n_tets, const GridGeom& g,
                                 double tet_mass, double* d_grid, DirectCounters* ctr, int device, hipStream_t stream) {
    return launch(LatticeTets{lat, pack_corners(corner_table(decomp)), d_ids}, n_tets, make_grid_desc(g, 0), tet_mass, d_grid,
                  ctr, device, stream);
}

hipError_t launch_direct_soup(const float* d_tets, int64_t n_tets, const GridGeom& g, double tet_mass, double* d_grid,
                              DirectCounters* ctr, int device, hipStream_t stream) {
    return launch(SoupTets{d_tets}, n_tets, make_grid_desc(g, 0), tet_mass, d_grid, ctr, device, stream);
}

hipError_t launch_direct_patches(const float* d_pos, int64_t num_patches, int m, int decomp, const GridGeom& g, double tet_mass,
                                 double* d_grid, DirectCounters* ctr, int device, hipStream_t stream) {
    return launch(PatchTets{d_pos, m, pack_corners(corner_table(decomp))}, num_patches * m * m * m * 6, make_grid_desc(g, 0),
                  tet_mass, d_grid, ctr, device, stream);
}

}  // namespace adeco
