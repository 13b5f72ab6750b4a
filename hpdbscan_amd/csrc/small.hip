// Clustering of small inputs by comparing all pairs of rows.
//
// The general path takes some 35 launches and four read-backs whatever the
// size: 2000 rows take 194 us, of which no kernel does work worth a launch.
// Without a sort and an index five kernels do (a row's sorted position is the
// number of rows with a smaller (cell, row), its candidates are the rows
// whose cell differs by at most one in every dimension):
//
//   k_small_grid    one block: min/max, the grid, every row's cell and key
//   k_small_count   all pairs: candidates, within-eps count and sorted
//                   position of every row, and the within-eps pairs as bits
//   k_small_hook    every core points at its neighbour core of smallest position
//   k_small_unite   union-find over the roots of those trees
//   k_small_label   cluster ids (roots), border and noise labels
//
// In k_small_count a block takes kRows rows and its 8 waves put 64 rows at a
// time against them, one per lane; the counts are population counts of
// ballots, and the ballots are the bit matrix.  The others take a row per wave
// and walk its bits.  Bound by the latency of a wave's chain of loads, hence
// the split over the waves of a block and the hook before the union-find:
// with every pair united directly, 1000 rows spent 47 us in chains of atomics.
// The results are those of the general path: the same cell index, the same
// squared distance, and a cluster's root is its smallest core position.
#include <algorithm>
#include <climits>

#include "boxes.hpp"
#include "cellkey.hpp"
#include "common.hpp"
#include "small.hpp"

namespace hpd {

namespace {

constexpr int kThreads = 512;
constexpr int kGridThreads = 1024;

// rows of a block: wave-uniform registers hold them
template <int D>
constexpr int kRows = D <= 4 ? 4 : 2;

// words of a bit per neighbour row of cells (3^(D-1) of them)
template <int D>
constexpr int row_words() {
    int r = 1;
    for (int j = 1; j < D; ++j) r *= 3;
    return (r + 31) / 32;
}

// 64-bit words of a row of the bit matrix
__host__ __device__ inline int64_t words_of(int64_t n) { return (n + 63) / 64; }

// What the kernels after the count read, whatever the rows' type.
struct SmallLinks {
    int32_t* pos;      // sorted position of every row
    int32_t* hook;     // by sorted position: the core pointed at (k_small_hook)
    int32_t* parent;   // by sorted position: union-find over the hooks' roots
    uint64_t* core;    // bit per row: core
    uint64_t* within;  // [n][words]: bit per row within eps (itself included)
};

template <typename T, int D>
struct SmallWork {
    uint64_t* key;    // cell id << sub_bits | sub-box digit
    int32_t* cell;    // cell index per swapped dimension, [n][D]
    SmallLinks l;
};

// eps2 and minPts: by value, or from the device's job table (a captured run is
// replayed with new ones)
template <typename T>
struct SmallParams {
    T eps2_v;
    uint32_t min_pts_v;
    const JobParams<T>* dev;
    __device__ __forceinline__ T eps2() const { return dev ? dev->eps2 : eps2_v; }
    __device__ __forceinline__ uint32_t min_pts() const { return dev ? dev->min_pts : min_pts_v; }
};

template <typename T, int D>
SmallWork<T, D> carve(void* work, int64_t n) {
    char* p = static_cast<char*>(work);
    auto take = [&](size_t bytes) {
        char* q = p;
        p += align_up(bytes, 256);
        return q;
    };
    const size_t nn = static_cast<size_t>(n);
    SmallWork<T, D> w;
    w.key = reinterpret_cast<uint64_t*>(take(8 * nn));
    w.cell = reinterpret_cast<int32_t*>(take(4 * D * nn));
    w.l.pos = reinterpret_cast<int32_t*>(take(4 * nn));
    w.l.hook = reinterpret_cast<int32_t*>(take(4 * nn));
    w.l.parent = reinterpret_cast<int32_t*>(take(4 * nn));
    w.l.core = reinterpret_cast<uint64_t*>(take(8 * static_cast<size_t>(words_of(n))));
    w.l.within = reinterpret_cast<uint64_t*>(take(8 * static_cast<size_t>(words_of(n)) * nn));
    return w;
}

template <typename T, int D>
__global__ __launch_bounds__(kGridThreads) void k_small_grid(const T* __restrict__ pts, int32_t n,
                                                             JobParams<T> jp,
                                                             const JobParams<T>* __restrict__ jp_dev,
                                                             int sub_k, int sub_bits,
                                                             SmallWork<T, D> w,
                                                             SmallResult* __restrict__ res) {
    if (jp_dev) jp = *jp_dev;
    constexpr int kGridWaves = kGridThreads / kWave;
    __shared__ T smn[kGridWaves][D], smx[kGridWaves][D];
    __shared__ alignas(16) unsigned char sjp_raw[sizeof(JobParams<T>)];
    JobParams<T>& sjp = *reinterpret_cast<JobParams<T>*>(sjp_raw);
    __shared__ int flags;  // 1: non-finite, 2: overflow, 4: unfit
    if (threadIdx.x == 0) flags = 0;
    T mn[D], mx[D];
#pragma unroll
    for (int k = 0; k < D; ++k) {
        mn[k] = min_init<T>();
        mx[k] = max_init<T>();
    }
    bool bad = false;
    for (int32_t i = static_cast<int32_t>(threadIdx.x); i < n; i += kGridThreads) {
#pragma unroll
        for (int k = 0; k < D; ++k) {
            const T c = pts[static_cast<int64_t>(i) * D + k];
            mn[k] = ref_min(mn[k], c);
            mx[k] = ref_max(mx[k], c);
            bad |= !isfinite(c);
        }
    }
    // NaN never wins the comparisons, so it is flagged by itself
    __syncthreads();
    if (__any(bad) && lane_id() == 0) atomicOr(&flags, 1);
#pragma unroll
    for (int k = 0; k < D; ++k) {
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) {
            mn[k] = ref_min(mn[k], __shfl_xor(mn[k], o, 64));
            mx[k] = ref_max(mx[k], __shfl_xor(mx[k], o, 64));
        }
        if (lane_id() == 0) {
            smn[threadIdx.x >> 6][k] = mn[k];
            smx[threadIdx.x >> 6][k] = mx[k];
        }
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        T mm[2 * D];
#pragma unroll
        for (int k = 0; k < D; ++k) {
            mm[k] = smn[0][k];
            mm[D + k] = smx[0][k];
            for (int v = 1; v < kGridWaves; ++v) {
                mm[k] = ref_min(mm[k], smn[v][k]);
                mm[D + k] = ref_max(mm[D + k], smx[v][k]);
            }
        }
        bool of = false;
        const uint64_t total = make_grid<T, D>(mm, jp, of);
        int f = of ? 2 : 0;
        const uint64_t maxkey = total - 1;
        const int bits = maxkey == 0 ? 0 : 64 - __clzll(static_cast<long long>(maxkey));
        if (bits + sub_bits > 64) f |= 4;
#pragma unroll
        for (int k = 0; k < D; ++k)
            if (jp.cp.ncell[k] > 0x7fffffffull) f |= 4;
        sjp = jp;
        if (f) atomicOr(&flags, f);
        SmallResult r = {};
        r.total_cells = total;
        const int all = flags;
        r.nonfinite = all & 1;
        r.overflow = (all >> 1) & 1;
        r.unfit = (all >> 2) & 1;
        *res = r;
    }
    __syncthreads();
    if (flags) return;
    for (int32_t i = static_cast<int32_t>(threadIdx.x); i < words_of(n); i += kGridThreads)
        w.l.core[i] = 0;
    for (int32_t i = static_cast<int32_t>(threadIdx.x); i < n; i += kGridThreads) {
        T row[D];
#pragma unroll
        for (int k = 0; k < D; ++k) row[k] = pts[static_cast<int64_t>(i) * D + k];
        w.key[i] = row_key<T, D>(row, sjp, sub_k, sub_bits);
#pragma unroll
        for (int k = 0; k < D; ++k) {
            const int j = sjp.cp.swapped[k];
            T x = row[0];
#pragma unroll
            for (int t = 1; t < D; ++t) x = t == j ? row[t] : x;
            w.cell[static_cast<int64_t>(i) * D + k] =
                static_cast<int32_t>(cell_index<T>(x, sjp.minv[j], jp.rcp_f, jp.rcp_d));
        }
    }
}

// Row q of the lane and whether its cell is a candidate cell of row p's.
template <typename T, int D>
__device__ __forceinline__ void load_small(const T* __restrict__ pts,
                                           const int32_t* __restrict__ cell, int32_t q, T* x,
                                           int32_t* c) {
#pragma unroll
    for (int k = 0; k < D; ++k) {
        x[k] = pts[static_cast<int64_t>(q) * D + k];
        c[k] = cell[static_cast<int64_t>(q) * D + k];
    }
}
template <int D>
__device__ __forceinline__ bool adjacent(const int32_t* a, const int32_t* b) {
    bool ok = true;
#pragma unroll
    for (int k = 0; k < D; ++k) ok = ok && static_cast<uint32_t>(a[k] - b[k] + 1) <= 2u;
    return ok;
}

__device__ __forceinline__ bool refused(const SmallResult* res) {
    return (res->nonfinite | res->overflow | res->unfit) != 0;
}

template <typename T, int D>
__global__ __launch_bounds__(kThreads) void k_small_count(const T* __restrict__ pts, int32_t n,
                                                          SmallParams<T> prm, int sub_bits,
                                                          SmallWork<T, D> w, SmallResult* res) {
    constexpr int R = kRows<D>;
    constexpr int W = row_words<D>();
    __shared__ uint32_t rows_lds[R][W];
    __shared__ uint32_t tot[R][3];  // candidates, within eps, sorted position
    __shared__ uint32_t seen[2];    // bit r: an earlier row shares row r's cell, box
    __shared__ unsigned long long sums[5];  // candidates, cores, cells, boxes, neighbour rows
    if (refused(res)) return;
    const T eps2 = prm.eps2();
    const uint32_t min_pts = prm.min_pts();
    const int t = static_cast<int>(threadIdx.x);
    if (t < 5) sums[t] = 0;
    if (t < 2) seen[t] = 0;
    if (t < R * 3) tot[t / 3][t % 3] = 0;
    for (int e = t; e < R * W; e += kThreads) rows_lds[e / W][e % W] = 0;
    const int32_t p0 = static_cast<int32_t>(blockIdx.x) * R;
    T xp[R][D];
    int32_t cp[R][D];
    uint64_t kp[R];
    uint32_t cand[R], cnt[R], pos[R];
    uint32_t seen_cell = 0, seen_box = 0;
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const int32_t p = min(p0 + r, n - 1);
        load_small<T, D>(pts, w.cell, p, xp[r], cp[r]);
        kp[r] = w.key[p];
        cand[r] = cnt[r] = pos[r] = 0;
    }
    __syncthreads();
    const int64_t words = words_of(n);
    for (int32_t q0 = uniform((t >> 6) * kWave); q0 < n; q0 += kThreads) {
        const int32_t q = min(q0 + lane_id(), n - 1);
        const bool in = q0 + lane_id() < n;
        T xq[D];
        int32_t cq[D];
        load_small<T, D>(pts, w.cell, q, xq, cq);
        const uint64_t kq = w.key[q];
#pragma unroll
        for (int r = 0; r < R; ++r) {
            const int32_t p = p0 + r;
            const bool adj = in && adjacent<D>(cp[r], cq);
            cand[r] += static_cast<uint32_t>(__popcll(ballot(adj)));
            const uint64_t near = ballot(adj && within<D>(xp[r], xq, eps2));
            cnt[r] += static_cast<uint32_t>(__popcll(near));
            if (lane_id() == 0 && p < n) w.l.within[p * words + (q0 >> 6)] = near;
            const uint64_t cellp = kp[r] >> sub_bits, cellq = kq >> sub_bits;
            const bool same = cellq == cellp && q < p;
            pos[r] += static_cast<uint32_t>(__popcll(ballot(in && (cellq < cellp || same))));
            if (__any(in && same)) seen_cell |= 1u << r;
            if (__any(in && kq == kp[r] && q < p)) seen_box |= 1u << r;
            // the neighbour rows of the cell (counted by its first row)
            if (!(seen_cell & (1u << r)) && adj) {
                int code = 0, mul = 1;
#pragma unroll
                for (int k = 1; k < D; ++k) {
                    code += (cq[k] - cp[r][k] + 1) * mul;
                    mul *= 3;
                }
                atomicOr(&rows_lds[r][code >> 5], 1u << (code & 31));
            }
        }
    }
    if (lane_id() == 0) {
#pragma unroll
        for (int r = 0; r < R; ++r) {
            atomicAdd(&tot[r][0], cand[r]);
            atomicAdd(&tot[r][1], cnt[r]);
            atomicAdd(&tot[r][2], pos[r]);
        }
        atomicOr(&seen[0], seen_cell);
        atomicOr(&seen[1], seen_box);
    }
    __syncthreads();
    // one wave per row
    const int r = t >> 6;
    if (r < R && p0 + r < n) {
        const bool is_core = tot[r][1] >= min_pts;
        const bool first = !(seen[0] & (1u << r));
        uint32_t rows = 0;
        if (first)
            for (int e = lane_id(); e < W; e += kWave)
                rows += static_cast<uint32_t>(__popc(rows_lds[r][e]));
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) rows += __shfl_xor(rows, o, 64);
        if (lane_id() == 0) {
            const int32_t at = static_cast<int32_t>(tot[r][2]);
            if (is_core)
                atomicOr(reinterpret_cast<unsigned long long*>(&w.l.core[(p0 + r) >> 6]),
                         1ull << ((p0 + r) & 63));
            w.l.pos[p0 + r] = at;
            atomicAdd(&sums[0], static_cast<unsigned long long>(tot[r][0]));
            if (is_core) atomicAdd(&sums[1], 1ull);
            if (first) {
                atomicAdd(&sums[2], 1ull);
                atomicAdd(&sums[4], static_cast<unsigned long long>(rows));
            }
            if (!(seen[1] & (1u << r))) atomicAdd(&sums[3], 1ull);
        }
    }
    __syncthreads();
    if (t < 5 && sums[t]) {
        unsigned long long* out[5] = {&res->sum_candidates, &res->cores, &res->cells, &res->boxes,
                                      &res->neighbor_rows};
        atomicAdd(out[t], sums[t]);
    }
}

// The row of the calling wave, one per wave of the grid.
constexpr int kRowThreads = 256;
template <int kBlock>
__device__ __forceinline__ int32_t wave_row() {
    return uniform(static_cast<int32_t>(blockIdx.x) * (kBlock / kWave) +
                   static_cast<int32_t>(threadIdx.x >> 6));
}
__device__ __forceinline__ bool is_core_row(const SmallLinks& l, int32_t p) {
    return (l.core[p >> 6] >> (p & 63)) & 1;
}
// place of the r-th set bit of m (r below their number)
__device__ __forceinline__ int nth_bit(uint64_t m, int r) {
    int at = 0;
#pragma unroll
    for (int w = 32; w > 0; w >>= 1) {
        const int c = __popcll(m & ((uint64_t{1} << w) - 1));
        const bool up = r >= c;
        r -= up ? c : 0;
        at += up ? w : 0;
        m = up ? m >> w : m;
    }
    return at;
}
// fn(on, q) for the cores q within eps of row p, 64 at a time, one per lane
// (`on`; q = p on the lanes beyond the last).  The row's words are read one
// per lane and the lanes share out their bits: the bits of one word at a time
// would be a few lanes and a chain of loads for each word.
template <typename Fn>
__device__ __forceinline__ void for_near_cores(const SmallLinks& l, int32_t n, int32_t p, Fn&& fn) {
    const int64_t words = words_of(n);
    const uint64_t* near = l.within + p * words;
    for (int64_t w0 = 0; w0 < words; w0 += kWave) {
        const int64_t wl = w0 + lane_id();
        const uint64_t mine = wl < words ? near[wl] & l.core[wl] : 0;
        const int bits = __popcll(mine);
        int incl = bits;
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) {
            const int t = __shfl_up(incl, o, 64);
            if (lane_id() >= o) incl += t;
        }
        const int excl = incl - bits;
        const int total = __builtin_amdgcn_readlane(incl, 63);
        for (int k0 = 0; k0 < total; k0 += kWave) {
            const int k = k0 + lane_id();
            int w = 0;  // the last word whose first bit is at or before k
#pragma unroll
            for (int st = 32; st > 0; st >>= 1)
                if (__shfl(excl, w + st, 64) <= k) w += st;
            const uint32_t lo = static_cast<uint32_t>(__shfl(static_cast<int>(mine), w, 64));
            const uint32_t hi = static_cast<uint32_t>(__shfl(static_cast<int>(mine >> 32), w, 64));
            const int first = __shfl(excl, w, 64);
            const bool on = k < total;
            const int bit = nth_bit((static_cast<uint64_t>(hi) << 32) | lo, on ? k - first : 0);
            fn(on, on ? static_cast<int32_t>(w0 + w) * kWave + bit : p);
        }
    }
}
// end of the chain v -> link[v] -> ... (links only lead down)
__device__ __forceinline__ int32_t chase(const int32_t* __restrict__ link, int32_t v) {
    for (int32_t next = link[v]; next != v; next = link[v]) v = next;
    return v;
}

// Every core points at its within-eps core of smallest sorted position (itself
// if that is its own): a forest whose roots are their trees' smallest members,
// and after which few pairs of cores have different roots.
__global__ __launch_bounds__(kRowThreads) void k_small_hook(int32_t n, SmallLinks l,
                                                            const SmallResult* res) {
    if (refused(res)) return;
    const int32_t p = wave_row<kRowThreads>();
    if (p >= n || !is_core_row(l, p)) return;
    int32_t first = INT_MAX;
    for_near_cores(l, n, p, [&](bool on, int32_t q) {
        if (on) first = min(first, l.pos[q]);
    });
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) first = min(first, __shfl_xor(first, o, 64));
    if (lane_id() == 0) {
        const int32_t pp = l.pos[p];
        l.hook[pp] = first;
        l.parent[pp] = pp;
    }
}

// The trees of within-eps cores joined: per row, lanes whose core is in the
// row's tree drop out, and one lane per remaining tree unites.
__global__ __launch_bounds__(kRowThreads) void k_small_unite(int32_t n, SmallLinks l,
                                                             const SmallResult* res) {
    if (refused(res)) return;
    const int32_t p = wave_row<kRowThreads>();
    if (p >= n || !is_core_row(l, p)) return;
    const int32_t pp = l.pos[p];
    const int32_t rp = chase(l.hook, pp);
    for_near_cores(l, n, p, [&](bool on, int32_t q) {
        const int32_t pq = l.pos[q];
        const int32_t rq = on && pq < pp ? chase(l.hook, pq) : rp;
        for (uint64_t todo = ballot(rq != rp); todo != 0;) {
            const int j = static_cast<int>(__builtin_ctzll(todo));
            const int32_t other = __builtin_amdgcn_readlane(rq, j);
            if (lane_id() == j) uf_unite(l.parent, rp, other);
            todo &= ~ballot(rq == other);
        }
    });
}

constexpr int kLabelThreads = 1024;
__global__ __launch_bounds__(kLabelThreads) void k_small_label(int32_t n, SmallLinks l,
                                                               SmallResult* res,
                                                               SmallResult* __restrict__ host,
                                                               int64_t* __restrict__ labels) {
    __shared__ unsigned int count[2];  // noise, ambiguous rows of the block
    __shared__ unsigned int done;
    if (threadIdx.x < 2) count[threadIdx.x] = 0;
    __syncthreads();
    const int32_t p = wave_row<kLabelThreads>();
    if (!refused(res) && p < n) {
        if (is_core_row(l, p)) {
            const int32_t c = chase(l.parent, chase(l.hook, l.pos[p]));
            if (lane_id() == 0) labels[p] = -(static_cast<int64_t>(c) + 1);
        } else {
            int32_t best = INT_MAX, worst = -1;  // smallest, largest adjacent cluster
            for_near_cores(l, n, p, [&](bool on, int32_t q) {
                if (!on) return;
                const int32_t c = chase(l.parent, chase(l.hook, l.pos[q]));
                best = min(best, c);
                worst = max(worst, c);
            });
#pragma unroll
            for (int o = 32; o > 0; o >>= 1) {
                best = min(best, __shfl_xor(best, o, 64));
                worst = max(worst, __shfl_xor(worst, o, 64));
            }
            if (lane_id() == 0) {
                labels[p] = best == INT_MAX ? 0 : static_cast<int64_t>(best) + 1;
                if (best == INT_MAX) atomicAdd(&count[0], 1u);
                else if (best != worst) atomicAdd(&count[1], 1u);
            }
        }
    }
    // the block that is done last hands the result to the host (its memory is
    // mapped; the caller waits for the stream before reading it)
    __syncthreads();
    if (threadIdx.x == 0) {
        if (count[0]) atomicAdd(&res->noise, static_cast<unsigned long long>(count[0]));
        if (count[1]) atomicAdd(&res->ambiguous, static_cast<unsigned long long>(count[1]));
        __threadfence();
        done = atomicAdd(&res->blocks_done, 1u);
        __threadfence();
    }
    __syncthreads();
    if (done + 1 == gridDim.x) {
        constexpr unsigned kWords = sizeof(SmallResult) / 4;
        if (threadIdx.x < kWords)
            reinterpret_cast<uint32_t*>(host)[threadIdx.x] =
                __hip_atomic_load(&reinterpret_cast<uint32_t*>(res)[threadIdx.x], __ATOMIC_RELAXED,
                                  __HIP_MEMORY_SCOPE_AGENT);
    }
}

}  // namespace

// All pairs against the general path, us, clouds of 60 blobs and (dense) of 5:
// 3-D float 2000 rows 69 / 194 and 91 / 214, 6000 148 / 211 and 170 / 196, 9000
// 242 / 228 and 282 / 197; 2-D 6000 155 / 213 and 192 / 202.  From 5-D on the
// general path's neighbourhoods grow with 3^D: 5-D float 7000 195 / 259 and 229 /
// 260, 9000 273 / 270 and 348 / 266 (double 7000 216 / 267 and 251 / 269); 6-D
// double 6000 187 / 295 and 238 / 307, 9000 328 / 330 and 387 / 337; 7-D float
// 9000 304 / 369 and 370 / 407, 11000 398 / 393 and 478 / 416 (double 9000 342 /
// 385 and 416 / 420); 8-D float 12000 477 / 903 and 643 / 721.
int64_t small_rows(int d) {
    switch (d) {
        case 5: return 7000;
        case 6: return 8000;
        case 7: return 10000;
        case 8: return 12000;
        default: return 6000;
    }
}

template <typename T, int D>
size_t small_workspace_bytes(int64_t n) {
    const size_t nn = static_cast<size_t>(n);
    const size_t words = static_cast<size_t>(words_of(n));
    return align_up(8 * nn, 256) + align_up(4 * D * nn, 256) + 3 * align_up(4 * nn, 256) +
           align_up(8 * words, 256) + align_up(8 * words * nn, 256);
}

template <typename T, int D>
void launch_small(const T* pts, int64_t n, const JobParams<T>& jp, const JobParams<T>* jp_dev,
                  int sub_k, int sub_bits, void* work, SmallResult* result, SmallResult* host,
                  int64_t* labels, hipStream_t s) {
    if (n <= 0) return;
    const int32_t nn = static_cast<int32_t>(n);
    const SmallWork<T, D> w = carve<T, D>(work, n);
    const SmallParams<T> prm{jp.eps2, jp.min_pts, jp_dev};
    const dim3 grid(static_cast<unsigned>((n + kRows<D> - 1) / kRows<D>));
    hipLaunchKernelGGL((k_small_grid<T, D>), dim3(1), dim3(kGridThreads), 0, s, pts, nn, jp, jp_dev,
                       sub_k, sub_bits, w, result);
    hipLaunchKernelGGL((k_small_count<T, D>), grid, dim3(kThreads), 0, s, pts, nn, prm, sub_bits, w,
                       result);
    auto rows = [&](int threads) {
        return dim3(static_cast<unsigned>((n * kWave + threads - 1) / threads));
    };
    hipLaunchKernelGGL(k_small_hook, rows(kRowThreads), dim3(kRowThreads), 0, s, nn, w.l,
                       static_cast<const SmallResult*>(result));
    hipLaunchKernelGGL(k_small_unite, rows(kRowThreads), dim3(kRowThreads), 0, s, nn, w.l,
                       static_cast<const SmallResult*>(result));
    hipLaunchKernelGGL(k_small_label, rows(kLabelThreads), dim3(kLabelThreads), 0, s, nn, w.l,
                       result, host, labels);
    HPD_HIP(hipGetLastError());
}

#define HPD_INST_SMALL(T, D)                                                                     \
    template size_t small_workspace_bytes<T, D>(int64_t);                                        \
    template void launch_small<T, D>(const T*, int64_t, const JobParams<T>&,                     \
                                     const JobParams<T>*, int, int, void*, SmallResult*,         \
                                     SmallResult*, int64_t*, hipStream_t);
#define HPD_INST_SMALL_ALL_D(T) \
    HPD_INST_SMALL(T, 1)        \
    HPD_INST_SMALL(T, 2)        \
    HPD_INST_SMALL(T, 3)        \
    HPD_INST_SMALL(T, 4)        \
    HPD_INST_SMALL(T, 5)        \
    HPD_INST_SMALL(T, 6)        \
    HPD_INST_SMALL(T, 7)        \
    HPD_INST_SMALL(T, 8)
HPD_INST_SMALL_ALL_D(float)
HPD_INST_SMALL_ALL_D(double)

}  // namespace hpd
