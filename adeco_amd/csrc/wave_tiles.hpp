// Device helpers shared by the persistent deposit kernels: the tiles of a candidate space as work
// items of a wavefront.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

#include "batched_impl.hpp"

namespace adeco {

__device__ __forceinline__ int upper_bound_i64(const int64_t* a, int n, int64_t v) {
    int lo = 0, hi = n;
    while (lo < hi) {
        const int mid = (lo + hi) >> 1;
        if (a[mid] <= v) lo = mid + 1;
        else hi = mid;
    }
    return lo;
}

__device__ __forceinline__ void wave_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

__device__ __forceinline__ int64_t shfl_i64(int64_t v, int src) {
    const int lo = __shfl(int(uint64_t(v) & 0xffffffffu), src, 64);
    const int hi = __shfl(int(uint64_t(v) >> 32), src, 64);
    return int64_t((uint64_t(unsigned(hi)) << 32) | unsigned(lo));
}

__device__ __forceinline__ int64_t shfl_up_i64(int64_t v, int d) {
    const int lo = __shfl_up(int(uint64_t(v) & 0xffffffffu), d, 64);
    const int hi = __shfl_up(int(uint64_t(v) >> 32), d, 64);
    return int64_t((uint64_t(unsigned(hi)) << 32) | unsigned(lo));
}

// What a tile's classification needs first: its source slot and index, its first pair, the number
// of pairs it touches and, per lane, the candidate offset of pair p0 + lane.  Loaded one tile
// ahead, so that these dependent loads overlap the previous tile's work.
struct TileHead {
    int slot;
    int p0, np;
    int64_t t;
    int64_t my_off;
};

template <class Sources>
__device__ __forceinline__ TileHead load_head(const Sources& srcs, const int2* __restrict__ entries, int64_t item,
                                              int lane) {
    TileHead h;
    h.slot = 0;
    h.t = item;
    if (entries) {
        const int2 en = entries[item];
        h.slot = __builtin_amdgcn_readfirstlane(en.x);
        h.t = int64_t(__builtin_amdgcn_readfirstlane(en.y));
    }
    const TileSource& src = srcs.get(h.slot);
    h.p0 = src.tile_first[h.t];
    h.np = min(src.tile_first[h.t + 1] - h.p0 + 1, kWaveTile);
    h.my_off = lane < h.np ? src.cand_off[h.p0 + lane] : int64_t(0);
    return h;
}

struct OneSource {
    TileSource s;
    __device__ const TileSource& get(int) const { return s; }
};
struct ManySources {
    const TileSource* s;
    __device__ const TileSource& get(int i) const { return s[i]; }
};

}  // namespace adeco
