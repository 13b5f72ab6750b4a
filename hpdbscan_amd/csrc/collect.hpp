// Collection of entries from a range of indices by the blocks of a grid, with one atomic per kCollectCap collected entries.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

#include "common.hpp"

namespace hpd {

constexpr int kCollectThreads = 256;
constexpr int kCollectWaves = kCollectThreads / kWave;
constexpr int kCollectPer = 2;  // indices per thread and round (100k rows, whole call
                                // in us: 1 309-317, 2 298-315, 4 325-330, 8 345)
constexpr int kCollectTile = kCollectThreads * kCollectPer;
constexpr int kCollectCap = 2048;  // entries staged in LDS

// The blocks take the tiles of [0, n) in turn, so that the blocks running
// together read and write one stretch of memory (with a slice of [0, n) per
// block the core labels' scattered writes of 4096 clouds took 5.2 ms, with
// tiles in turn 2.7).  One reservation per scanned tile would be an atomic on
// one address per 512 slots (10M rows: 20k of them); staged, it is one per
// 2048 entries found.
constexpr unsigned kCollectBlocks = 2048;
inline unsigned collect_blocks(int64_t n) {
    const int64_t t = (n + kCollectTile - 1) / kCollectTile;
    return static_cast<unsigned>(t < kCollectBlocks ? (t > 0 ? t : 1) : kCollectBlocks);
}

// fn(i, v) is called once for every index of the block's tiles (by one
// thread each); where it returns true, v goes to out[..], in index order
// inside a tile; *count grows by the number of entries.  Every thread of
// a block of kCollectThreads calls it.
template <typename E, typename Fn>
__device__ __forceinline__ void block_collect(int64_t n, E* __restrict__ out,
                                              unsigned int* __restrict__ count, Fn&& fn) {
    __shared__ E buf[kCollectCap];
    __shared__ unsigned int wcnt[kCollectWaves];
    __shared__ unsigned int at;
    const int w = static_cast<int>(threadIdx.x >> 6);
    unsigned int fill = 0;  // equal in every thread
    auto flush = [&] {
        if (threadIdx.x == 0) at = atomicAdd(count, fill);
        __syncthreads();
        const unsigned int base = at;
        for (unsigned int e = threadIdx.x; e < fill; e += kCollectThreads) out[base + e] = buf[e];
        __syncthreads();
        fill = 0;
    };
    for (int64_t t = static_cast<int64_t>(blockIdx.x) * kCollectTile; t < n;
         t += static_cast<int64_t>(gridDim.x) * kCollectTile) {
        uint64_t m[kCollectPer];
        E v[kCollectPer];
        unsigned int c = 0;
#pragma unroll
        for (int k = 0; k < kCollectPer; ++k) {
            const int64_t i = t + w * (kWave * kCollectPer) + k * kWave + lane_id();
            m[k] = ballot(i < n && fn(i, v[k]));
            c += static_cast<unsigned int>(__popcll(m[k]));
        }
        if (lane_id() == 0) wcnt[w] = c;
        __syncthreads();
        unsigned int off = 0, tot = 0;
#pragma unroll
        for (int k = 0; k < kCollectWaves; ++k) {
            if (k < w) off += wcnt[k];
            tot += wcnt[k];
        }
        if (fill + tot > kCollectCap) flush();
        off += fill;
        const uint64_t lt = lanemask_lt();
#pragma unroll
        for (int k = 0; k < kCollectPer; ++k) {
            if ((m[k] >> lane_id()) & 1ull) buf[off + __popcll(m[k] & lt)] = v[k];
            off += static_cast<unsigned int>(__popcll(m[k]));
        }
        fill += tot;
        __syncthreads();
    }
    if (fill) flush();
}

}  // namespace hpd
