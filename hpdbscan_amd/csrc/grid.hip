// eps-grid construction on the device:
//   k_minmax_partial / k_minmax_final  per-dimension min and max
//                                      (spatial_index.h:99-122, with the
//                                      reference's initial values :531-532)
//   k_cell_ids                         linearised cell id of every row
//                                      (spatial_index.h:144-165)
//   k_gather_soa                       coordinates in sorted order, one
//                                      array per dimension
#include <cfloat>
#include <limits>
#include <type_traits>

#include "cellkey.hpp"
#include "common.hpp"
#include "grid.hpp"
#include "internal.hpp"

namespace hpd {

namespace {

constexpr int kMMThreads = 256;
constexpr int kMMRows = 8 * kMMThreads;  // rows per partial block, at least
// the final pass is one block per job: a job's partials stay below this
constexpr int64_t kMMBlocks = 2048;

// One block reduces up to `rpb` rows of one job; bfirst[j] is the first block
// of job j (one job: rows [row0, row1), jobs and bfirst not read).
template <typename T, int D>
__global__ __launch_bounds__(kMMThreads) void k_minmax_partial(
    const T* __restrict__ pts, int64_t row0, int64_t row1, const JobParams<T>* __restrict__ jobs,
    int32_t njobs, const int32_t* __restrict__ bfirst, int64_t rpb, T* __restrict__ part,
    int* __restrict__ bad_part) {
    const int32_t b = static_cast<int32_t>(blockIdx.x);
    int64_t r0 = row0 + b * rpb, r1 = row1;
    if (njobs > 1) {
        const int32_t j = wave_last(njobs, [&](int32_t k) { return bfirst[k] <= b; });
        r0 = jobs[j].row_begin + (b - bfirst[j]) * rpb;
        r1 = jobs[j].row_end;
    }
    r1 = min(r0 + rpb, r1);
    T mn[D], mx[D];
#pragma unroll
    for (int k = 0; k < D; ++k) {
        mn[k] = min_init<T>();
        mx[k] = max_init<T>();
    }
    bool bad = false;
    for (int64_t i = r0 + threadIdx.x; i < r1; i += kMMThreads) {
#pragma unroll
        for (int k = 0; k < D; ++k) {
            const T c = pts[i * D + k];
            mn[k] = ref_min(mn[k], c);
            mx[k] = ref_max(mx[k], c);
            if constexpr (std::is_floating_point<T>::value) bad |= !isfinite(c);
        }
    }
    // NaN never wins the comparisons above, so non-finite input is flagged
    // separately (the host rejects it)
    const int any_bad = __syncthreads_or(bad ? 1 : 0);
    __shared__ T smn[D][kMMThreads];
    __shared__ T smx[D][kMMThreads];
#pragma unroll
    for (int k = 0; k < D; ++k) {
        smn[k][threadIdx.x] = mn[k];
        smx[k][threadIdx.x] = mx[k];
    }
    __syncthreads();
    for (int o = kMMThreads / 2; o > 0; o >>= 1) {
        if (threadIdx.x < o) {
#pragma unroll
            for (int k = 0; k < D; ++k) {
                smn[k][threadIdx.x] = ref_min(smn[k][threadIdx.x], smn[k][threadIdx.x + o]);
                smx[k][threadIdx.x] = ref_max(smx[k][threadIdx.x], smx[k][threadIdx.x + o]);
            }
        }
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        bad_part[b] = any_bad;
#pragma unroll
        for (int k = 0; k < D; ++k) {
            part[static_cast<int64_t>(b) * 2 * D + k] = smn[k][0];
            part[static_cast<int64_t>(b) * 2 * D + D + k] = smx[k][0];
        }
    }
}

// One block per job: min/max over the job's partial blocks; *nonfinite |= 1 (one
// job: stored) when a row is not finite.  out and nonfinite may be pinned host
// memory for one job.
template <typename T, int D>
__global__ __launch_bounds__(kMMThreads) void k_minmax_final(const T* __restrict__ part,
                                                             const int* __restrict__ bad_part,
                                                             const int32_t* __restrict__ bfirst,
                                                             int32_t njobs, int32_t nblocks,
                                                             T* __restrict__ out,
                                                             int* __restrict__ nonfinite) {
    const int32_t j = static_cast<int32_t>(blockIdx.x);
    const int32_t b0 = njobs == 1 ? 0 : bfirst[j];
    const int32_t b1 = njobs == 1 ? nblocks : bfirst[j + 1];
    int bad = 0;
    __shared__ T smn[D][kMMThreads];
    __shared__ T smx[D][kMMThreads];
    T mn[D], mx[D];
#pragma unroll
    for (int k = 0; k < D; ++k) {
        mn[k] = min_init<T>();
        mx[k] = max_init<T>();
    }
    for (int32_t b = b0 + static_cast<int32_t>(threadIdx.x); b < b1; b += kMMThreads) {
        bad |= bad_part[b];
#pragma unroll
        for (int k = 0; k < D; ++k) {
            mn[k] = ref_min(mn[k], part[static_cast<int64_t>(b) * 2 * D + k]);
            mx[k] = ref_max(mx[k], part[static_cast<int64_t>(b) * 2 * D + D + k]);
        }
    }
#pragma unroll
    for (int k = 0; k < D; ++k) {
        smn[k][threadIdx.x] = mn[k];
        smx[k][threadIdx.x] = mx[k];
    }
    bad = __syncthreads_or(bad);
    for (int o = kMMThreads / 2; o > 0; o >>= 1) {
        if (threadIdx.x < o) {
#pragma unroll
            for (int k = 0; k < D; ++k) {
                smn[k][threadIdx.x] = ref_min(smn[k][threadIdx.x], smn[k][threadIdx.x + o]);
                smx[k][threadIdx.x] = ref_max(smx[k][threadIdx.x], smx[k][threadIdx.x + o]);
            }
        }
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        if (njobs == 1) *nonfinite = bad ? 1 : 0;
        else if (bad) atomicOr(nonfinite, 1);
#pragma unroll
        for (int k = 0; k < D; ++k) {
            out[static_cast<int64_t>(j) * 2 * D + k] = smn[k][0];
            out[static_cast<int64_t>(j) * 2 * D + D + k] = smx[k][0];
        }
    }
}

// A wave takes kIdRows consecutive rows.
constexpr int kIdRows = 256;
template <typename T, int D, typename K>
__global__ __launch_bounds__(256) void k_cell_ids(const T* __restrict__ pts, int64_t n,
                                                  const JobParams<T>* __restrict__ jobs,
                                                  int32_t njobs, int sub_k, int sub_bits,
                                                  K* __restrict__ keys,
                                                  uint32_t* __restrict__ vals) {
    const int64_t r0 = (static_cast<int64_t>(blockIdx.x) * 4 + (threadIdx.x >> 6)) * kIdRows;
    for_job_rows(jobs, njobs, r0, r0 + kIdRows < n ? r0 + kIdRows : n,
                 [&](const JobParams<T>& jp, int64_t i) {
        keys[i] = static_cast<K>(row_key<T, D>(pts + i * D, jp, sub_k, sub_bits));
        vals[i] = static_cast<uint32_t>(i);
    });
}

template <typename T>
__global__ __launch_bounds__(256) void k_put_job(const JobParams<T> v, JobParams<T>* __restrict__ dst,
                                                 uint32_t* __restrict__ zero, int nzero) {
    if (threadIdx.x == 0) *dst = v;
    for (int i = threadIdx.x; i < nzero; i += 256) zero[i] = 0u;
}

template <typename T, int D>
__global__ __launch_bounds__(256) void k_gather_soa(const T* __restrict__ pts, int64_t n,
                                                    const uint32_t* __restrict__ order,
                                                    T* __restrict__ soa, int64_t ld) {
    const int64_t i = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
    if (i >= n) return;
    const int64_t o = order[i];
#pragma unroll
    for (int j = 0; j < D; ++j) soa[static_cast<int64_t>(j) * ld + i] = pts[o * D + j];
}

// The grid of every job from its min / max (mm: 2D values per job), as the
// host computes it after reading them back (make_grid); then key bases in job
// order.  flags[0] |= 1: a grid of more than 2^64 cells; *sort_bits = bits
// of the largest key + sub_bits; *total = all jobs' cells.  One block.
template <typename T, int D>
__global__ __launch_bounds__(256) void k_geometry(JobParams<T>* __restrict__ jobs, int32_t njobs,
                                                  const T* __restrict__ mm, int sub_bits,
                                                  uint64_t* __restrict__ cells,
                                                  int* __restrict__ flags,
                                                  int* __restrict__ sort_bits,
                                                  unsigned long long* __restrict__ total) {
    __shared__ unsigned long long part[256];
    __shared__ int bad;
    if (threadIdx.x == 0) bad = 0;
    __syncthreads();
    // per job: geometry and number of cells (0 for a job without rows)
    for (int32_t j = threadIdx.x; j < njobs; j += 256) {
        JobParams<T>& jp = jobs[j];
        uint64_t tot = 0;
        if (jp.row_end > jp.row_begin) {
            bool of = false;
            tot = make_grid<T, D>(&mm[static_cast<int64_t>(j) * 2 * D], jp, of);
            if (of) atomicOr(&bad, 1);
        }
        cells[j] = tot;
    }
    __syncthreads();
    // key bases: each thread sums a contiguous run of jobs, the runs are
    // scanned, then every thread assigns its run's bases
    const int32_t per = (njobs + 255) / 256;
    const int32_t j0 = static_cast<int32_t>(threadIdx.x) * per;
    const int32_t j1 = min(njobs, j0 + per);
    unsigned long long sum = 0;
    bool of = false;
    for (int32_t j = j0; j < j1; ++j) of |= __builtin_add_overflow(sum, cells[j], &sum);
    part[threadIdx.x] = sum;
    if (of) atomicOr(&bad, 1);
    __syncthreads();
    if (threadIdx.x == 0) {
        unsigned long long acc = 0;
        bool o2 = false;
        for (int t = 0; t < 256; ++t) {
            const unsigned long long v = part[t];
            part[t] = acc;
            o2 |= __builtin_add_overflow(acc, v, &acc);
        }
        if (o2) bad = 1;
        *total = acc;
        const uint64_t maxkey = acc > 0 ? acc - 1 : 0;
        const int kb = maxkey == 0 ? 0 : 64 - __clzll(static_cast<long long>(maxkey));
        *sort_bits = kb + sub_bits;
        if (kb + sub_bits > 64) bad = 1;
    }
    __syncthreads();
    unsigned long long base = part[threadIdx.x];
    for (int32_t j = j0; j < j1; ++j) {
        jobs[j].key_base = base;
        base += cells[j];
    }
    if (threadIdx.x == 0 && bad) flags[0] |= 1;
}

inline unsigned blocks_for(int64_t n, int t) { return static_cast<unsigned>((n + t - 1) / t); }

// out[i] = in[i] as float; four values per thread, the block's loads of one
// round side by side (no alignment of `in` beyond its own type's)
template <typename T>
__global__ __launch_bounds__(256) void k_to_float(const T* __restrict__ in, int64_t count,
                                                  float* __restrict__ out) {
    const int64_t i0 = static_cast<int64_t>(blockIdx.x) * 1024 + threadIdx.x;
#pragma unroll
    for (int k = 0; k < 4; ++k)
        if (i0 + k * 256 < count) out[i0 + k * 256] = static_cast<float>(in[i0 + k * 256]);
}

}  // namespace

template <typename T, int D>
void launch_geometry(JobParams<T>* jobs, int32_t njobs, const T* mm, int sub_bits, uint64_t* cells,
                     int* flags, int* sort_bits, unsigned long long* total, hipStream_t s) {
    hipLaunchKernelGGL((k_geometry<T, D>), dim3(1), dim3(256), 0, s, jobs, njobs, mm, sub_bits, cells,
                       flags, sort_bits, total);
    HPD_HIP(hipGetLastError());
}

int64_t minmax_rows_per_block(int64_t n) {
    const int64_t per = static_cast<int64_t>(kMMRows) * kMMBlocks;
    return kMMRows * (n > per ? (n + per - 1) / per : 1);
}

template <typename T>
void launch_put_job(const JobParams<T>& v, JobParams<T>* dst, void* zero, size_t zero_bytes,
                    hipStream_t s) {
    hipLaunchKernelGGL(k_put_job<T>, dim3(1), dim3(256), 0, s, v, dst, static_cast<uint32_t*>(zero),
                       static_cast<int>(zero_bytes / 4));
    HPD_HIP(hipGetLastError());
}

template <typename T>
void launch_to_float(const T* in, int64_t count, float* out, hipStream_t s) {
    if (count <= 0) return;
    hipLaunchKernelGGL(k_to_float<T>, dim3(blocks_for((count + 3) / 4, 256)), dim3(256), 0, s, in,
                       count, out);
    HPD_HIP(hipGetLastError());
}

template <typename T, int D>
void launch_minmax(const T* pts, int64_t row0, int64_t row1, const JobParams<T>* jobs,
                   int32_t njobs, const int32_t* bfirst, int32_t nblocks, int64_t rpb, T* part,
                   int* bad_part, T* out, int* nonfinite, hipStream_t s) {
    if (nblocks > 0)
        hipLaunchKernelGGL((k_minmax_partial<T, D>), dim3(nblocks), dim3(kMMThreads), 0, s, pts,
                           row0, row1, jobs, njobs, bfirst, rpb, part, bad_part);
    hipLaunchKernelGGL((k_minmax_final<T, D>), dim3(njobs), dim3(kMMThreads), 0, s,
                       static_cast<const T*>(part), static_cast<const int*>(bad_part), bfirst,
                       njobs, nblocks, out, nonfinite);
    HPD_HIP(hipGetLastError());
}

template <typename T, int D, typename K>
void launch_cell_ids(const T* pts, int64_t n, const JobParams<T>* jobs, int32_t njobs, int sub_k,
                     int sub_bits, K* keys, uint32_t* vals, hipStream_t s) {
    if (n <= 0) return;
    hipLaunchKernelGGL((k_cell_ids<T, D, K>), dim3(blocks_for(n, 4 * kIdRows)), dim3(256), 0, s, pts, n,
                       jobs, njobs, sub_k, sub_bits, keys, vals);
    HPD_HIP(hipGetLastError());
}

template <typename T, int D>
void launch_gather_soa(const T* pts, int64_t n, const uint32_t* order, T* soa, int64_t ld,
                       hipStream_t s) {
    if (n <= 0) return;
    hipLaunchKernelGGL((k_gather_soa<T, D>), dim3(blocks_for(n, 256)), dim3(256), 0, s, pts, n,
                       order, soa, ld);
    HPD_HIP(hipGetLastError());
}

#define HPD_INST_GRID(T, D)                                                                     \
    template void launch_geometry<T, D>(JobParams<T>*, int32_t, const T*, int, uint64_t*, int*,  \
                                        int*, unsigned long long*, hipStream_t);                  \
    template void launch_minmax<T, D>(const T*, int64_t, int64_t, const JobParams<T>*, int32_t,  \
                                      const int32_t*, int32_t, int64_t, T*, int*, T*, int*,      \
                                      hipStream_t);                                              \
    template void launch_cell_ids<T, D, uint32_t>(const T*, int64_t, const JobParams<T>*,        \
                                                  int32_t, int, int, uint32_t*, uint32_t*,       \
                                                  hipStream_t);                                  \
    template void launch_cell_ids<T, D, uint64_t>(const T*, int64_t, const JobParams<T>*,        \
                                                  int32_t, int, int, uint64_t*, uint32_t*,       \
                                                  hipStream_t);                                  \
    template void launch_gather_soa<T, D>(const T*, int64_t, const uint32_t*, T*, int64_t,      \
                                          hipStream_t);

#define HPD_INST_GRID_ALL_D(T) \
    HPD_INST_GRID(T, 1)        \
    HPD_INST_GRID(T, 2)        \
    HPD_INST_GRID(T, 3)        \
    HPD_INST_GRID(T, 4)        \
    HPD_INST_GRID(T, 5)        \
    HPD_INST_GRID(T, 6)        \
    HPD_INST_GRID(T, 7)        \
    HPD_INST_GRID(T, 8)

HPD_FOR_EACH_DTYPE(HPD_INST_GRID_ALL_D)

#define HPD_INST_TO_FLOAT(T) template void launch_to_float<T>(const T*, int64_t, float*, hipStream_t);
HPD_FOR_EACH_DTYPE(HPD_INST_TO_FLOAT)

#define HPD_INST_PUT_JOB(T) \
    template void launch_put_job<T>(const JobParams<T>&, JobParams<T>*, void*, size_t, hipStream_t);
HPD_FOR_EACH_DTYPE(HPD_INST_PUT_JOB)

}  // namespace hpd
