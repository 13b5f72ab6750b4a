// Streaming candidate rows through a wave: the rows are read in aligned
// batches with wave-uniform addresses (a few wide scalar loads per batch),
// every lane tests its own row against each candidate of the batch.
#pragma once

#include <hip/hip_runtime.h>

#include <climits>
#include <cstdint>
#include <type_traits>

#include "common.hpp"

namespace hpd {

template <typename T, int D>
__device__ __forceinline__ void load_row(const T* __restrict__ soa, int64_t ld, int64_t i, T* c) {
#pragma unroll
    for (int j = 0; j < D; ++j) c[j] = soa[static_cast<int64_t>(j) * ld + i];
}

// Candidates are visited in aligned batches of kBatch<T> rows.  Every batch
// is fetched with wave-uniform addresses before it is used, which lets the
// compiler issue them as a few wide scalar loads and wait once.
template <typename T>
constexpr int kBatch = sizeof(T) == 8 ? 8 : 16;

template <typename U, int B>
struct alignas(B * sizeof(U) >= 4 ? B * sizeof(U) : 4) Batch {
    U v[B];
};

template <typename U, int B>
__device__ __forceinline__ Batch<U, B> load_batch(const U* __restrict__ base, int64_t a) {
    return *reinterpret_cast<const Batch<U, B>*>(base + a);
}

// Visit candidate rows [qb, qe).  body(q, qc, core_q, aux_q) runs per
// candidate; core_q is flags[q] (1 without flags), aux_q is aux[q] (0 without
// aux).  stop() is checked after each batch and ends the visit when true.
// Returns true if stopped.  soa, flags and aux are read up to the next
// multiple of the batch size past qe (callers pad them to ld rows).
template <typename T, int D, typename Body, typename Stop>
__device__ __forceinline__ bool visit_range(const T* __restrict__ soa, int64_t ld,
                                            const uint8_t* __restrict__ flags,
                                            const int32_t* __restrict__ aux, int32_t qb, int32_t qe,
                                            Body&& body, Stop&& stop) {
    constexpr int B = kBatch<T>;
    for (int32_t a = qb & ~(B - 1); a < qe; a += B) {
        Batch<T, B> b[D];
#pragma unroll
        for (int j = 0; j < D; ++j) b[j] = load_batch<T, B>(soa + static_cast<int64_t>(j) * ld, a);
        Batch<uint8_t, B> f;
        if (flags) f = load_batch<uint8_t, B>(flags, a);
        Batch<int32_t, B> x;
        if (aux) x = load_batch<int32_t, B>(aux, a);
        const bool full = a >= qb && a + B <= qe;
        const int lo = qb > a ? qb - a : 0;
        const int hi = qe - a < B ? qe - a : B;
#pragma unroll
        for (int t = 0; t < B; ++t) {
            if (!full && (t < lo || t >= hi)) continue;
            T qc[D];
#pragma unroll
            for (int j = 0; j < D; ++j) qc[j] = b[j].v[t];
            body(a + t, qc, flags ? f.v[t] : uint8_t(1), aux ? x.v[t] : 0);
        }
        if (stop()) return true;
    }
    return false;
}

// order-preserving integer images of floating-point values (for atomics)
__device__ __forceinline__ uint32_t ord_key(float f) {
    const uint32_t u = __float_as_uint(f);
    return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}
__device__ __forceinline__ float ord_val(uint32_t k) {
    return __uint_as_float((k & 0x80000000u) ? (k & 0x7fffffffu) : ~k);
}
__device__ __forceinline__ unsigned long long ord_key(double f) {
    const unsigned long long u = static_cast<unsigned long long>(__double_as_longlong(f));
    return (u & 0x8000000000000000ull) ? ~u : (u | 0x8000000000000000ull);
}
__device__ __forceinline__ double ord_val(unsigned long long k) {
    return __longlong_as_double(static_cast<long long>((k & 0x8000000000000000ull)
                                                           ? (k & 0x7fffffffffffffffull)
                                                           : ~k));
}

template <typename T>
using OrdKey = std::conditional_t<sizeof(T) == 8, unsigned long long, uint32_t>;

// Bounding box of a box in one dimension: bbox[b * D + j].
template <typename T>
struct alignas(2 * sizeof(T)) Span {
    T lo, hi;
};

// Bounds of the reference's squared distance between a row and the members
// of a box: gmin2 <= dist2(p, q) <= gmax2 for every member q, where gmin2 and
// gmax2 are the reference's own expression (sum2) on the differences to the
// box's nearest and farthest point.  Every step of it (subtract, square, each
// add of the summation tree, the flush of tiny values) rounds monotonically,
// so the bounds hold for the rounded values themselves: gmin2 > EPS2 rules
// every member out and gmax2 <= EPS2 rules every member in, with no margin.
template <typename T, int D>
__device__ __forceinline__ void point_box(const Span<T>* __restrict__ bbox, int32_t b, const T* pc,
                                          T& gmin2, T& gmax2) {
    T g[D], f[D];
#pragma unroll
    for (int j = 0; j < D; ++j) {
        const Span<T> s = bbox[static_cast<int64_t>(b) * D + j];
        const T below = s.lo - pc[j], above = pc[j] - s.hi;
        g[j] = max(T(0), max(below, above));
        f[j] = max(-below, -above);
    }
    gmin2 = sum2<D>(g);
    gmax2 = sum2<D>(f);
}

// Wave-uniform copy of lane j's value (j wave-uniform): v_readlane.
__device__ __forceinline__ int32_t bcast(int32_t v, int j) {
    return __builtin_amdgcn_readlane(v, j);
}
__device__ __forceinline__ uint64_t bcast64(uint64_t v, int j) {
    const uint32_t lo = static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(v), j));
    const uint32_t hi = static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(v >> 32), j));
    return (static_cast<uint64_t>(hi) << 32) | lo;
}
__device__ __forceinline__ double bcast(double v, int j) {
    const long long x = __double_as_longlong(v);
    const uint32_t lo = static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(x), j));
    const uint32_t hi =
        static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(x >> 32), j));
    return __longlong_as_double(static_cast<long long>((static_cast<uint64_t>(hi) << 32) | lo));
}

__device__ __forceinline__ float bcast(float v, int j) {
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), j));
}

// Candidates on the lanes: how many of the rows [qb, qe) (with flags: of
// those whose flag is set) are within eps of the wave-uniform row pr, counted
// until the count reaches `limit` (a look after every kWideStep rows; the
// result is exact below the limit and at least the limit otherwise).
// visit_range reads 16 candidates an iteration for up to 64 rows at once;
// with a few rows that leaves the lanes idle and a box of a million rows is
// one wave's chain of 65k dependent iterations.  Here an iteration reads
// kWideStep rows, coalesced.  visited += rows read.
constexpr int kWideLoads = 4;
constexpr int kWideStep = 64 * kWideLoads;
// Rows of a wave up to which a box of more than kWideMinRows rows is walked
// row by row with the candidates on the lanes: an iteration of either walk
// costs about one load latency and 16 x 4 tests, so 256 candidates of one
// row cost what 16 candidates of all 64 do.  One-wave chains were the whole
// core count of 100M skewed 2-D rows (7.85 ms for 2.3M tests).
constexpr int kWideRows = 8;
constexpr int kWideMinRows = 64;

template <typename T, int D>
__device__ __forceinline__ uint32_t wide_count(const T* __restrict__ soa, int64_t ld,
                                               const uint8_t* __restrict__ flags, int32_t qb,
                                               int32_t qe, const T* pr, T eps2, uint32_t limit,
                                               uint32_t& visited) {
    uint32_t cnt = 0;
    const int lane = __lane_id();
    for (int32_t a = qb; a < qe && cnt < limit; a += kWideStep) {
        T c[kWideLoads][D];
        uint8_t f[kWideLoads];
#pragma unroll
        for (int k = 0; k < kWideLoads; ++k) {
            const int32_t q = min(a + k * 64 + lane, qe - 1);
            load_row<T, D>(soa, ld, q, c[k]);
            f[k] = flags ? flags[q] : uint8_t(1);
        }
#pragma unroll
        for (int k = 0; k < kWideLoads; ++k) {
            const bool in = a + k * 64 + lane < qe && f[k] && within<D>(pr, c[k], eps2);
            cnt += static_cast<uint32_t>(__popcll(__ballot(in)));
        }
        visited += static_cast<uint32_t>(min(kWideStep, qe - a));
    }
    return cnt;
}

// The rows of the lanes in `rows` walked as above; true on the lanes whose
// row has a candidate (with flags: a flagged one) within eps.
template <typename T, int D>
__device__ __forceinline__ bool wide_any(const T* __restrict__ soa, int64_t ld,
                                         const uint8_t* __restrict__ flags, int32_t qb, int32_t qe,
                                         const T* pc, T eps2, uint64_t rows, bool first_only) {
    bool hit = false;
    uint32_t visited = 0;
    for (; rows != 0; rows &= rows - 1) {
        const int r = static_cast<int>(__builtin_ctzll(rows));
        T pr[D];
#pragma unroll
        for (int e = 0; e < D; ++e) pr[e] = bcast(pc[e], r);
        const bool h = wide_count<T, D>(soa, ld, flags, qb, qe, pr, eps2, 1u, visited) != 0;
        if (__lane_id() == r) hit = h;
        if (h && first_only) break;
    }
    return hit;
}

// Whether a walk of n candidate rows for the lanes of `rows` goes row by row.
__device__ __forceinline__ bool walk_wide(uint64_t rows, int32_t n) {
    return n > kWideMinRows && __popcll(rows) <= kWideRows;
}

// A wave split into groups of G lanes, each with a neighbourhood of its own:
// the boxes of the neighbour rows [r0, r1) of an occupied cell (box ranges
// rboxes, the own row `center` first, from the cell's first box `own` on and
// wrapping round, then the other rows in stored order) are handed out G at a
// time, one per lane.  fn(valid, b) runs for the whole wave at once (it may
// use wave-wide operations), with the lane's box b where valid; what it
// returns must be equal over a group: true ends that group's visit.  Only
// boxes in [bmin, bmax) are visited.  All arguments but G are per lane, equal over
// a group; inactive groups take part in the wave-wide steps only.
//
// Why groups: a neighbourhood holds some 10-30 boxes, so a whole wave per
// row, box or cell leaves most lanes without one, and a thread per row or box
// walks them as a chain of dependent loads.
template <int G, typename Fn>
__device__ __forceinline__ void group_boxes(bool active, int32_t r0, int32_t r1, int32_t center,
                                            int32_t own, const int2* __restrict__ rboxes,
                                            int32_t bmin, int32_t bmax, Fn&& fn) {
    const int gl = __lane_id() & (G - 1);
    const int32_t nrows = r1 - r0;
    for (int32_t g0 = 0; __any(active && g0 < nrows); g0 += G) {
        // G rows at a time, one per lane
        const int32_t i = g0 + gl;
        int32_t b0 = 0, cnt = 0;
        if (active && i < nrows) {
            const int32_t r = i == 0 ? center : (r0 + i - 1 < center ? r0 + i - 1 : r0 + i);
            const int2 bs = rboxes[r];
            b0 = max(bs.x, bmin);
            cnt = max(0, min(bs.y, bmax) - b0);
        }
        // the own row starts at box `own`
        const int32_t rot = g0 == 0 && gl == 0 && own > b0 && own < b0 + cnt ? own - b0 : 0;
        int32_t incl = cnt;
#pragma unroll
        for (int o = 1; o < G; o <<= 1) {
            const int32_t t = __shfl_up(incl, o, G);
            if (gl >= o) incl += t;
        }
        const int32_t excl = incl - cnt;
        const int32_t total = __shfl(incl, G - 1, G);
        const int32_t rot0 = __shfl(rot, 0, G);
        const int32_t n0 = __shfl(cnt, 0, G);
        for (int32_t k0 = 0; __any(active && k0 < total); k0 += G) {
            const int32_t kk = k0 + gl;
            int32_t row = 0;  // the last row whose first box is at or before kk
#pragma unroll
            for (int st = G / 2; st > 0; st >>= 1) {
                const int32_t e = __shfl(excl, row + st, G);
                if (e <= kk) row += st;
            }
            int32_t local = kk - __shfl(excl, row, G);
            if (g0 == 0 && row == 0) local += local + rot0 < n0 ? rot0 : rot0 - n0;
            const int32_t b = __shfl(b0, row, G) + local;
            if (fn(active && kk < total, b)) active = false;
        }
    }
}

// Lanes (and rows) per chunk of the core count, and the rows of a box up to
// which the box's lane walks it by itself.  Lanes: neighbourhoods grow with
// 3^D (core count, ms: 5M rows of 4 (16 lanes) 0.55, (32) 0.444; 30k of 6
// doubles (16) 0.110, (32) 0.078).
template <int D>
constexpr int kGroup = D <= 3 ? 8 : 32;
constexpr int kLaneRows = 8;

// Persistent grids: wave w of them takes items w, w + wave_stride(), ...
// Workgroups go to the 8 XCDs in turn, and each XCD has an L2 of its own, so
// the waves are numbered XCD by XCD: of the stretch of items that the grid
// works on together, each XCD takes one eighth, and neighbouring items, which
// read the same boxes, meet in one L2.
constexpr int kGroupThreads = 256;
constexpr unsigned kXcds = 8;
__device__ __forceinline__ int32_t first_wave() {
    unsigned blk = blockIdx.x;
    if (gridDim.x % kXcds == 0) blk = (blk % kXcds) * (gridDim.x / kXcds) + blk / kXcds;
    return __builtin_amdgcn_readfirstlane(static_cast<int32_t>(blk) * (kGroupThreads / 64) +
                                          static_cast<int32_t>(threadIdx.x >> 6));
}
__device__ __forceinline__ int32_t wave_stride() {
    return static_cast<int32_t>(gridDim.x) * (kGroupThreads / 64);
}
// Blocks of one over at most `items` items, `per_wave` per wave: no more than
// run at once (every block then starts at once, and none is left to run by
// itself after the others), a multiple of the XCDs when there are that many.
template <auto Kernel>
inline unsigned persistent_blocks(int64_t items, int per_wave) {
    static const int64_t resident = [] {
        int dev = 0, cus = 0, per_cu = 0;
        if (hipGetDevice(&dev) != hipSuccess ||
            hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess ||
            hipOccupancyMaxActiveBlocksPerMultiprocessor(
                &per_cu, reinterpret_cast<const void*>(Kernel), kGroupThreads, 0) != hipSuccess ||
            cus < 1 || per_cu < 1)
            return int64_t{2048};
        return static_cast<int64_t>(cus) * per_cu;
    }();
    const int64_t per_block = static_cast<int64_t>(per_wave) * (kGroupThreads / 64);
    int64_t b = (items + per_block - 1) / per_block;
    if (b > resident) b = resident;
    if (b >= kXcds) b -= b % kXcds;
    return static_cast<unsigned>(b > 0 ? b : 1);
}

// Orders the LDS accesses of a wave's lanes among each other (the hardware
// keeps a wave's LDS operations in order; this keeps the compiler from moving
// or caching them).
__device__ __forceinline__ void wave_lds_fence() {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
}

// Sum, minimum and maximum over a group of G lanes.
template <int G>
__device__ __forceinline__ uint32_t group_sum(uint32_t v) {
#pragma unroll
    for (int o = G / 2; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    return v;
}
template <int G>
__device__ __forceinline__ int32_t group_min(int32_t v) {
#pragma unroll
    for (int o = G / 2; o > 0; o >>= 1) v = min(v, __shfl_xor(v, o, 64));
    return v;
}
template <int G>
__device__ __forceinline__ int32_t group_max(int32_t v) {
#pragma unroll
    for (int o = G / 2; o > 0; o >>= 1) v = max(v, __shfl_xor(v, o, 64));
    return v;
}

// Runs of equal `key` over consecutive lanes (boxes are contiguous slot
// ranges): afterwards every lane holds the minimum (maximum) of v over the
// lanes from itself to the end of its run.
template <typename U>
__device__ __forceinline__ U run_suffix_min(U v, int32_t key) {
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const U w = __shfl_down(v, o, 64);
        const int32_t k = __shfl_down(key, o, 64);
        if (__lane_id() + o < 64 && k == key) v = w < v ? w : v;
    }
    return v;
}
template <typename U>
__device__ __forceinline__ U run_suffix_max(U v, int32_t key) {
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const U w = __shfl_down(v, o, 64);
        const int32_t k = __shfl_down(key, o, 64);
        if (__lane_id() + o < 64 && k == key) v = w > v ? w : v;
    }
    return v;
}

// True on the lane holding the first slot of its run of equal `key`.
__device__ __forceinline__ bool run_head(int32_t key) {
    const int32_t prev = __shfl_up(key, 1, 64);
    return __lane_id() == 0 || prev != key;
}

}  // namespace hpd
