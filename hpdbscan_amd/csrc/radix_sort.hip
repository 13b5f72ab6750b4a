// Stable LSD radix sort of (cell id, row index) pairs, 8 or 9 bits per pass.
//
// Replaces the reference's cell histogram + serial counting-sort scatter
// (spatial_index.h:144-216).  Per pass:
//   1. k_radix_hist    digit histogram of every block's run of tiles
//   2. exclusive scan  of the histograms -> global offset of (digit, block);
//                      for few blocks each block of 3. adds them up itself
//   3. k_radix_scatter stable rank of every key inside its tile (wave
//                      ballots + per-wave LDS counters), the tile staged
//                      in LDS in digit order, then written out so that
//                      consecutive threads write consecutive places
// A tile is 4096 keys: 4 waves x 16 iterations x 64 lanes (fewer iterations for
// few keys); the stable order inside a tile is (wave, iteration, lane), i.e.
// input order.  9-bit digits
// (512 buckets, two per thread) are used where they save a pass.
//
// A block takes a run of tiles (SortPlan) where there are more than
// kRunBlocks of them: with one tile per block the histograms of 100M keys are
// 50 MB per pass, written, scanned and read back in single words.  Longer runs
// save more there but leave too few blocks to hide a tile's chain of barriers
// (100M rows, 2 passes, sort phase in ms by the blocks left: 2048 4.05, 4096
// 4.10, 8192 3.93, 16384 3.87, all 48828 3.98).
#include <type_traits>

#include "common.hpp"
#include "hpdbscan_capi.h"
#include "internal.hpp"

namespace hpd {

namespace {

constexpr int kThreads = 256;
constexpr int kIters = 16;
// passes that carry rows stage them in LDS too: half the tile keeps two
// more blocks resident per CU
constexpr int kItersRows = 8;
constexpr int kItersMin = 4;
constexpr int kMaxBuckets = 512;          // 9-bit digits

__host__ __device__ inline int64_t tiles_of(int64_t n, int64_t tile) {
    return (n + tile - 1) / tile;
}

// How a sort of n keys splits: blocks of `run` tiles of kThreads * iters keys;
// with self, each scatter block adds up the histograms (hist[block * buckets +
// digit], written and read in rows) instead of a scan of hist[digit * blocks +
// block]: two launches fewer per pass for up to kSelfBlocks * 1 KB read by
// every block.  Where that is so the tiles are the smallest that leave no more
// than kSelfBlocks of them: a tile's ranking is a serial chain of its
// iterations, and 100k rows fill 25 of 256 CUs with tiles of 4096 (sort phase,
// tiles of 4096 against this rule: 100k rows of 3 floats 126 -> 102 us, 30k of 6
// doubles 159 -> 109, 200k of 3 136 -> 117; with up to 768 blocks 102, 110, 113).
constexpr int64_t kRunBlocks = 16384;
constexpr int64_t kSelfBlocks = 192;
struct SortPlan {
    int64_t blocks;
    int iters;
    int run;
    bool self;
};
// (9-bit digits from 2048 keys on: half the blocks, so that no plan needs more
// histogram words than kMaxBuckets per 2048 keys)
inline SortPlan sort_plan(int64_t n, int max_iters, int bits) {
    int iters = bits > 8 ? 2 * kItersMin : kItersMin;
    while (iters < max_iters && tiles_of(n, kThreads * iters) > kSelfBlocks) iters *= 2;
    const int64_t tiles = tiles_of(n, kThreads * iters);
    const int64_t run = tiles_of(tiles, kRunBlocks);
    const int64_t blocks = tiles_of(tiles, run);
    return SortPlan{blocks, iters, static_cast<int>(run), blocks <= kSelfBlocks};
}
// fn(std::integral_constant<int, iters>)
template <int kMax, typename Fn>
void with_iters(const SortPlan& plan, Fn&& fn) {
    static_assert(kMax == 8 || kMax == 16, "the iterations of a full tile");
    if (plan.iters == 4) fn(std::integral_constant<int, 4>{});
    else if (plan.iters == 8) fn(std::integral_constant<int, 8>{});
    else fn(std::integral_constant<int, kMax>{});
}

template <typename K, int kBits, int kIt>
__global__ __launch_bounds__(kThreads) void k_radix_hist(const K* __restrict__ keys, int64_t n,
                                                         int shift, uint32_t* __restrict__ hist,
                                                         SortPlan plan,
                                                         const int* __restrict__ bits_dev) {
    if (bits_dev && shift >= *bits_dev) return;  // a pass beyond the key's bits
    constexpr int B = 1 << kBits;
    constexpr uint32_t kMask = B - 1;
    __shared__ uint32_t cnt[B];
    for (int dg = threadIdx.x; dg < B; dg += kThreads) cnt[dg] = 0;
    __syncthreads();
    constexpr int tile = kThreads * kIt;
    const int64_t base = static_cast<int64_t>(blockIdx.x) * plan.run * tile;
    const int64_t end = base + static_cast<int64_t>(plan.run) * tile;
    const int64_t stop = end < n ? end : n;
    for (int64_t t = base + threadIdx.x; t < stop; t += tile) {
        K k[kIt];
#pragma unroll
        for (int it = 0; it < kIt; ++it) {
            const int64_t idx = t + it * kThreads;
            k[it] = idx < stop ? keys[idx] : K(0);
        }
#pragma unroll
        for (int it = 0; it < kIt; ++it)
            if (t + it * kThreads < stop)
                atomicAdd(&cnt[static_cast<uint32_t>((k[it] >> shift) & kMask)], 1u);
    }
    __syncthreads();
    for (int dg = threadIdx.x; dg < B; dg += kThreads) {
        if (plan.self)
            hist[static_cast<int64_t>(blockIdx.x) * B + dg] = cnt[dg];
        else
            hist[static_cast<int64_t>(dg) * plan.blocks + blockIdx.x] = cnt[dg];
    }
}

// Rows that a pass carries along with the pairs: row i of `in` (one word W
// of D values of T) goes where pair i goes, into `out` (words), or on the
// last pass into D planes of stride ld (the coordinates in sorted order).
// The row is read with its key, staged in LDS with it and written with it.
struct NoRows {
    static constexpr bool kOn = false;
    using W = uint32_t;
    __device__ W load(int64_t) const { return 0; }
    __device__ void store(int64_t, W) const {}
};
template <typename T, int D>
struct MoveRows {
    static constexpr bool kOn = true;
    using W = std::conditional_t<sizeof(T) * D == 8, uint64_t, uint32_t>;
    static_assert(sizeof(T) * D == sizeof(W), "a row is one 4- or 8-byte word");
    const W* in;
    W* out;      // ld == 0
    T* planes;   // ld > 0
    int64_t ld;
    __device__ __forceinline__ W load(int64_t i) const { return in[i]; }
    __device__ __forceinline__ void store(int64_t to, W v) const {
        if (ld > 0) {
            T x[D];
            __builtin_memcpy(x, &v, sizeof(W));
#pragma unroll
            for (int j = 0; j < D; ++j) planes[static_cast<int64_t>(j) * ld + to] = x[j];
        } else {
            out[to] = v;
        }
    }
};

template <typename K, int kBits, int kIt, typename Rows = NoRows>
__global__ __launch_bounds__(kThreads) void k_radix_scatter(const K* __restrict__ kin,
                                                            const uint32_t* __restrict__ vin,
                                                            K* __restrict__ kout,
                                                            uint32_t* __restrict__ vout, int64_t n,
                                                            int shift,
                                                            const uint32_t* __restrict__ offs,
                                                            SortPlan plan,
                                                            const int* __restrict__ bits_dev,
                                                            Rows rows = Rows{}) {
    if (bits_dev && shift >= *bits_dev) return;  // a pass beyond the key's bits
    constexpr int B = 1 << kBits;
    constexpr uint32_t kMask = B - 1;
    constexpr int kOwn = B / kThreads;  // consecutive digits per thread
    __shared__ uint32_t cnt[4][B];
    __shared__ uint32_t gbase[B];
    __shared__ uint32_t tbase[B];  // digit's first place in the staged tile
    __shared__ uint32_t wsum[kThreads / 64];
    constexpr int tile = kThreads * kIt;
    __shared__ K skey[tile];
    __shared__ uint32_t sval[tile];
    __shared__ typename Rows::W srow[Rows::kOn ? tile : 1];
    const int w = threadIdx.x >> 6;
    const int l = threadIdx.x & 63;
    if (plan.self) {
        // Own offset of a digit: its keys in earlier blocks (gbase) plus all
        // keys of smaller digits (from tbase).  The waves take the blocks'
        // histograms in turn, four digits per lane and load.
        constexpr int kQ = B / 256;
        constexpr int kDeep = 8;  // rows in flight per wave
        for (int dg = threadIdx.x; dg < B; dg += kThreads) gbase[dg] = tbase[dg] = 0;
        uint4 before[kQ], all[kQ];
#pragma unroll
        for (int q = 0; q < kQ; ++q) before[q] = all[q] = make_uint4(0, 0, 0, 0);
        const uint4* rows4 = reinterpret_cast<const uint4*>(offs);
        const int nblk = static_cast<int>(plan.blocks);
        for (int b = w; b < nblk; b += 4 * kDeep) {
            uint4 v[kDeep][kQ];
#pragma unroll
            for (int j = 0; j < kDeep; ++j)
#pragma unroll
                for (int q = 0; q < kQ; ++q)
                    v[j][q] = b + 4 * j < nblk ? rows4[(b + 4 * j) * (B / 4) + q * 64 + l]
                                               : make_uint4(0, 0, 0, 0);
#pragma unroll
            for (int j = 0; j < kDeep; ++j)
#pragma unroll
                for (int q = 0; q < kQ; ++q) {
                    const uint32_t in = b + 4 * j < static_cast<int>(blockIdx.x) ? ~0u : 0u;
                    before[q].x += v[j][q].x & in;
                    before[q].y += v[j][q].y & in;
                    before[q].z += v[j][q].z & in;
                    before[q].w += v[j][q].w & in;
                    all[q].x += v[j][q].x;
                    all[q].y += v[j][q].y;
                    all[q].z += v[j][q].z;
                    all[q].w += v[j][q].w;
                }
        }
        __syncthreads();
#pragma unroll
        for (int q = 0; q < kQ; ++q) {
            const int dg = q * 256 + 4 * l;
            atomicAdd(&gbase[dg], before[q].x);
            atomicAdd(&gbase[dg + 1], before[q].y);
            atomicAdd(&gbase[dg + 2], before[q].z);
            atomicAdd(&gbase[dg + 3], before[q].w);
            atomicAdd(&tbase[dg], all[q].x);
            atomicAdd(&tbase[dg + 1], all[q].y);
            atomicAdd(&tbase[dg + 2], all[q].z);
            atomicAdd(&tbase[dg + 3], all[q].w);
        }
        __syncthreads();
        uint32_t below = 0;  // keys of the digits of earlier rounds
#pragma unroll
        for (int o = 0; o < kOwn; ++o) {
            const uint32_t sum = tbase[o * kThreads + threadIdx.x];
            uint32_t inc = sum;
#pragma unroll
            for (int st = 1; st < 64; st <<= 1) {
                const uint32_t t = __shfl_up(inc, st, 64);
                if (l >= st) inc += t;
            }
            if (l == 63) wsum[w] = inc;
            __syncthreads();
            uint32_t woff = 0, total = 0;
#pragma unroll
            for (int i = 0; i < kThreads / 64; ++i) {
                if (i < w) woff += wsum[i];
                total += wsum[i];
            }
            gbase[o * kThreads + threadIdx.x] += below + woff + inc - sum;
            below += total;
            __syncthreads();
        }
    } else {
        for (int dg = threadIdx.x; dg < B; dg += kThreads)
            gbase[dg] = offs[static_cast<int64_t>(dg) * plan.blocks + blockIdx.x];
    }
    const int64_t run0 = static_cast<int64_t>(blockIdx.x) * plan.run * tile;
    for (int r = 0; r < plan.run; ++r) {
        const int64_t tile0 = run0 + static_cast<int64_t>(r) * tile;
        if (tile0 >= n) break;
        for (int dg = threadIdx.x; dg < B; dg += kThreads) {
#pragma unroll
            for (int i = 0; i < 4; ++i) cnt[i][dg] = 0;
        }
        __syncthreads();

        const int64_t base = tile0 + w * (tile / 4);
        const uint64_t lt = lanemask_lt();
        K key[kIt];
        uint32_t val[kIt];
        uint32_t rank[kIt];
        uint32_t dgt[kIt];
        typename Rows::W row[Rows::kOn ? kIt : 1];
#pragma unroll
        for (int it = 0; it < kIt; ++it) {
            const int64_t idx = base + it * 64 + l;
            const bool valid = idx < n;
            const K k = valid ? kin[idx] : K(0);
            const uint32_t d = static_cast<uint32_t>((k >> shift) & kMask);
            uint64_t peers = ballot(valid);
#pragma unroll
            for (int b = 0; b < kBits; ++b) {
                const bool bit = (d >> b) & 1u;
                const uint64_t m = ballot(bit);
                peers &= bit ? m : ~m;
            }
            uint32_t c = 0;
            if (valid) c = cnt[w][d];
            if (valid && (peers & lt) == 0) cnt[w][d] = c + static_cast<uint32_t>(__popcll(peers));
            rank[it] = c + static_cast<uint32_t>(__popcll(peers & lt));
            dgt[it] = valid ? d : 0xffffffffu;
            key[it] = k;
            val[it] = valid ? vin[idx] : 0u;
            if constexpr (Rows::kOn) row[it] = valid ? rows.load(idx) : 0;
        }
        __syncthreads();
        // exclusive prefix of each digit over the four waves, and of the digits'
        // tile totals over the digits (thread t owns digits [t * kOwn, ..))
        uint32_t tot[kOwn];
        uint32_t run = 0;
#pragma unroll
        for (int o = 0; o < kOwn; ++o) {
            const int dg = threadIdx.x * kOwn + o;
            uint32_t acc = 0;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const uint32_t c = cnt[i][dg];
                cnt[i][dg] = acc;
                acc += c;
            }
            tot[o] = acc;
            run += acc;
        }
        uint32_t inc = run;
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) {
            const uint32_t t = __shfl_up(inc, o, 64);
            if (l >= o) inc += t;
        }
        if (l == 63) wsum[w] = inc;
        __syncthreads();
        uint32_t woff = 0;
#pragma unroll
        for (int i = 0; i < kThreads / 64; ++i)
            if (i < w) woff += wsum[i];
        uint32_t first = woff + inc - run;
#pragma unroll
        for (int o = 0; o < kOwn; ++o) {
            tbase[threadIdx.x * kOwn + o] = first;
            first += tot[o];
        }
        __syncthreads();
        // stage the tile in digit order (stable: waves, iterations and lanes are
        // in input order) ...
#pragma unroll
        for (int it = 0; it < kIt; ++it) {
            if (dgt[it] != 0xffffffffu) {
                const uint32_t at = tbase[dgt[it]] + cnt[w][dgt[it]] + rank[it];
                skey[at] = key[it];
                sval[at] = val[it];
                if constexpr (Rows::kOn) srow[at] = row[it];
            }
        }
        __syncthreads();
        // ... and write it out: consecutive threads write consecutive places of
        // one digit's run
        const int64_t left = n - tile0;
        const int valid_in_tile = left < tile ? static_cast<int>(left) : tile;
#pragma unroll
        for (int it = 0; it < kIt; ++it) {
            const int at = it * kThreads + threadIdx.x;
            if (at < valid_in_tile) {
                const K k = skey[at];
                const uint32_t d = static_cast<uint32_t>((k >> shift) & kMask);
                const uint32_t dst = gbase[d] + (static_cast<uint32_t>(at) - tbase[d]);
                kout[dst] = k;
                vout[dst] = sval[at];
                if constexpr (Rows::kOn) rows.store(dst, srow[at]);
            }
        }
        __syncthreads();
        // the next tile's keys go after this one's
#pragma unroll
        for (int o = 0; o < kOwn; ++o) gbase[threadIdx.x * kOwn + o] += tot[o];
    }
}

// After passes beyond a device-written bit count did nothing, the result of
// the `launched` passes lies in the b buffers when an odd number of them ran:
// copy it back to the a buffers.
template <typename K>
__global__ __launch_bounds__(kThreads) void k_radix_settle(K* __restrict__ keys_a,
                                                           uint32_t* __restrict__ vals_a,
                                                           const K* __restrict__ keys_b,
                                                           const uint32_t* __restrict__ vals_b,
                                                           int64_t n, int digit_bits,
                                                           const int* __restrict__ bits_dev) {
    const int ran = (*bits_dev + digit_bits - 1) / digit_bits;
    if ((ran & 1) == 0) return;
    for (int64_t i = static_cast<int64_t>(blockIdx.x) * kThreads + threadIdx.x; i < n;
         i += static_cast<int64_t>(gridDim.x) * kThreads) {
        keys_a[i] = keys_b[i];
        vals_a[i] = vals_b[i];
    }
}

template <typename K, int kBits>
bool sort_passes(K* keys_a, uint32_t* vals_a, K* keys_b, uint32_t* vals_b, int64_t n, int bits,
                 uint32_t* hist, uint32_t* tmp, hipStream_t s, const int* bits_dev = nullptr) {
    const SortPlan plan = sort_plan(n, kIters, kBits);
    const dim3 grid(static_cast<unsigned>(plan.blocks));
    K* kin = keys_a;
    uint32_t* vin = vals_a;
    K* kout = keys_b;
    uint32_t* vout = vals_b;
    bool in_b = false;
    for (int shift = 0; shift < bits; shift += kBits) {
        with_iters<kIters>(plan, [&](auto iters) {
            constexpr int kIt = decltype(iters)::value;
            hipLaunchKernelGGL((k_radix_hist<K, kBits, kIt>), grid, dim3(kThreads), 0, s, kin, n,
                               shift, hist, plan, bits_dev);
            if (!plan.self) exclusive_scan_u32(hist, hist, plan.blocks << kBits, tmp, nullptr, s);
            hipLaunchKernelGGL((k_radix_scatter<K, kBits, kIt>), grid, dim3(kThreads), 0, s, kin,
                               vin, kout, vout, n, shift, hist, plan, bits_dev);
        });
        HPD_HIP(hipGetLastError());
        K* tk = kin;
        kin = kout;
        kout = tk;
        uint32_t* tv = vin;
        vin = vout;
        vout = tv;
        in_b = !in_b;
    }
    return in_b;
}

// sort_passes carrying rows: pass 0 reads them from `pts`, passes in
// between alternate between rows_a and rows_b, the last writes the planes
template <typename K, int kBits, typename T, int D>
bool sort_passes_rows(K* keys_a, uint32_t* vals_a, K* keys_b, uint32_t* vals_b, int64_t n,
                      int bits, uint32_t* hist, uint32_t* tmp, const T* pts, T* rows_a,
                      T* rows_b, T* soa, int64_t ld, hipStream_t s) {
    const SortPlan plan = sort_plan(n, kItersRows, kBits);
    const dim3 grid(static_cast<unsigned>(plan.blocks));
    K* kin = keys_a;
    uint32_t* vin = vals_a;
    K* kout = keys_b;
    uint32_t* vout = vals_b;
    bool in_b = false;
    const T* rin = pts;
    T* rnext = rows_a;
    for (int shift = 0; shift < bits; shift += kBits) {
        const bool last = shift + kBits >= bits;
        using W = typename MoveRows<T, D>::W;
        MoveRows<T, D> mv{reinterpret_cast<const W*>(rin), reinterpret_cast<W*>(rnext), soa,
                          last ? ld : 0};
        with_iters<kItersRows>(plan, [&](auto iters) {
            constexpr int kIt = decltype(iters)::value;
            hipLaunchKernelGGL((k_radix_hist<K, kBits, kIt>), grid, dim3(kThreads), 0, s, kin, n,
                               shift, hist, plan, nullptr);
            if (!plan.self) exclusive_scan_u32(hist, hist, plan.blocks << kBits, tmp, nullptr, s);
            hipLaunchKernelGGL((k_radix_scatter<K, kBits, kIt, MoveRows<T, D>>), grid,
                               dim3(kThreads), 0, s, kin, vin, kout, vout, n, shift, hist, plan,
                               nullptr, mv);
        });
        HPD_HIP(hipGetLastError());
        K* tk = kin;
        kin = kout;
        kout = tk;
        uint32_t* tv = vin;
        vin = vout;
        vout = tv;
        in_b = !in_b;
        rin = rnext;
        rnext = rnext == rows_a ? rows_b : rows_a;
    }
    return in_b;
}

}  // namespace

int radix_pass_count(int bits) {
    if (bits <= 0) return 0;
    const int digit = (bits + 8) / 9 < (bits + 7) / 8 ? 9 : 8;
    return (bits + digit - 1) / digit;
}

size_t radix_hist_words(int64_t n) {
    return static_cast<size_t>(kMaxBuckets) *
           static_cast<size_t>(tiles_of(n > 0 ? n : 1, kThreads * kItersRows));
}

// 9-bit digits where they save a pass (e.g. 25-27 key bits: 3 passes, not 4)
template <typename K>
bool radix_sort_pairs(K* keys_a, uint32_t* vals_a, K* keys_b, uint32_t* vals_b, int64_t n,
                      int bits, uint32_t* hist, uint32_t* tmp, hipStream_t s) {
    if (n <= 1 || bits <= 0) return false;
    if ((bits + 8) / 9 < (bits + 7) / 8)
        return sort_passes<K, 9>(keys_a, vals_a, keys_b, vals_b, n, bits, hist, tmp, s);
    return sort_passes<K, 8>(keys_a, vals_a, keys_b, vals_b, n, bits, hist, tmp, s);
}

template <typename K, typename T, int D>
bool radix_sort_pairs_rows(K* keys_a, uint32_t* vals_a, K* keys_b, uint32_t* vals_b, int64_t n,
                           int bits, uint32_t* hist, uint32_t* tmp, const T* pts, T* rows_a,
                           T* rows_b, T* soa, int64_t ld, hipStream_t s) {
    if (n <= 1 || bits <= 0)
        throw Error(HPD_EINVAL, "radix_sort_pairs_rows needs n > 1 and bits > 0");
    if ((bits + 8) / 9 < (bits + 7) / 8)
        return sort_passes_rows<K, 9, T, D>(keys_a, vals_a, keys_b, vals_b, n, bits, hist, tmp,
                                            pts, rows_a, rows_b, soa, ld, s);
    return sort_passes_rows<K, 8, T, D>(keys_a, vals_a, keys_b, vals_b, n, bits, hist, tmp, pts,
                                        rows_a, rows_b, soa, ld, s);
}

#define HPD_INST_SORT_ROWS(K, T, D)                                                              \
    template bool radix_sort_pairs_rows<K, T, D>(K*, uint32_t*, K*, uint32_t*, int64_t, int,     \
                                                 uint32_t*, uint32_t*, const T*, T*, T*, T*,     \
                                                 int64_t, hipStream_t);
#define HPD_INST_SORT_ROWS_K(T, D) HPD_INST_SORT_ROWS(uint32_t, T, D) HPD_INST_SORT_ROWS(uint64_t, T, D)
HPD_INST_SORT_ROWS_K(float, 1)
HPD_INST_SORT_ROWS_K(float, 2)
HPD_INST_SORT_ROWS_K(double, 1)

template <typename K>
void radix_sort_pairs_dev(K* keys_a, uint32_t* vals_a, K* keys_b, uint32_t* vals_b, int64_t n,
                          int max_bits, const int* bits_dev, uint32_t* hist, uint32_t* tmp,
                          hipStream_t s) {
    if (n <= 1 || max_bits <= 0) return;
    sort_passes<K, 8>(keys_a, vals_a, keys_b, vals_b, n, max_bits, hist, tmp, s, bits_dev);
    const int64_t want = (n + kThreads - 1) / kThreads;
    hipLaunchKernelGGL(k_radix_settle<K>, dim3(static_cast<unsigned>(want < 4096 ? want : 4096)),
                       dim3(kThreads), 0, s, keys_a, vals_a, static_cast<const K*>(keys_b),
                       static_cast<const uint32_t*>(vals_b), n, 8, bits_dev);
    HPD_HIP(hipGetLastError());
}

template void radix_sort_pairs_dev<uint64_t>(uint64_t*, uint32_t*, uint64_t*, uint32_t*, int64_t,
                                             int, const int*, uint32_t*, uint32_t*, hipStream_t);

template bool radix_sort_pairs<uint32_t>(uint32_t*, uint32_t*, uint32_t*, uint32_t*, int64_t, int,
                                         uint32_t*, uint32_t*, hipStream_t);
template bool radix_sort_pairs<uint64_t>(uint64_t*, uint32_t*, uint64_t*, uint32_t*, int64_t, int,
                                         uint32_t*, uint32_t*, hipStream_t);

}  // namespace hpd
