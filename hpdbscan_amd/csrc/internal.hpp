// Host-side declarations shared by the translation units of the library.
#pragma once

#include <hip/hip_runtime.h>

#include <cstddef>
#include <cstdint>
#include <stdexcept>
#include <type_traits>
#include <string>
#include <vector>

namespace hpd {

constexpr int kMaxDims = 8;  // dimensions handled by the device kernels

// An error carrying an hpd_status code; the C-ABI layer turns it into the
// return value and the thread-local message.
struct Error : std::runtime_error {
    int code;
    Error(int c, const std::string& m) : std::runtime_error(m), code(c) {}
};

void check_hip(hipError_t e, const char* what);
#define HPD_HIP(call) ::hpd::check_hip((call), #call)

// Grow-only device arena.  Allocations are 256-byte aligned bump pointers
// into one hipMalloc'd block; reset() recycles the block for the next call.
// An arena attached to memory it does not own never allocates: reserve()
// beyond its capacity throws HPD_EUNSUPPORTED.
class Arena {
public:
    Arena() = default;
    ~Arena();
    Arena(const Arena&) = delete;
    Arena& operator=(const Arena&) = delete;

    // Use [base, base + cap) (256-byte aligned) instead of allocating.
    void attach(void* base, size_t cap) {
        base_ = static_cast<char*>(base);
        cap_ = cap;
        used_ = 0;
        owned_ = false;
    }
    // Make sure at least `bytes` are available in one block (drops contents).
    void reserve(size_t bytes);
    // Give an allocation of its own back.
    void release();
    void reset() { used_ = 0; }
    void* take(size_t bytes);
    template <typename T>
    T* take_n(size_t n) {
        return static_cast<T*>(take(n * sizeof(T)));
    }
    size_t capacity() const { return cap_; }
    const void* base() const { return base_; }
    size_t used() const { return used_; }

private:
    char* base_ = nullptr;
    size_t cap_ = 0;
    size_t used_ = 0;
    bool owned_ = true;
};

inline size_t align_up(size_t x, size_t a) { return (x + a - 1) / a * a; }

// A number of items known on the host, or (dev not null) written into device
// memory by an earlier kernel, `host` being then an upper bound that sizes
// the launch (tight: a bound close to the count, such as the number of boxes
// for a list of boxes, rather than a worst case).  The static pipeline (no
// host read-backs) passes the latter throughout, the plain one for lists
// whose length it does not wait for.
struct Count {
    int64_t host = 0;
    const uint32_t* dev = nullptr;
    bool tight = false;  // host is close to the count: one wave per item of it
    __device__ __forceinline__ int64_t get() const {
        return dev ? static_cast<int64_t>(*dev) : host;
    }
};
inline Count host_count(int64_t n) { return Count{n, nullptr}; }

// Exclusive prefix sum of n uint32 values (in may equal out).  `tmp` must
// hold scan_tmp_words(n) uint32.  The total is written to *total_dev when
// total_dev is not null (device memory).
size_t scan_tmp_words(int64_t n);
void exclusive_scan_u32(const uint32_t* in, uint32_t* out, int64_t n, uint32_t* tmp,
                        uint32_t* total_dev, hipStream_t s);
// The same over a length that an earlier kernel wrote (n.dev, at most
// n.host, which sizes the launches); the total goes to out[length].
void exclusive_scan_u32_dev(const uint32_t* in, uint32_t* out, Count n, uint32_t* tmp,
                            hipStream_t s);
// *dst = a[*idx_dev] (a scan's total at a device-written length, moved to a
// fixed place)
void copy_at_count(const uint32_t* a, const uint32_t* idx_dev, uint32_t* dst, hipStream_t s);
// *dst[i] = *src[i] for i < k (device words)
struct WordCopies {
    const uint32_t* src[8];
    uint32_t* dst[8];
    int k = 0;
    void add(const uint32_t* from, uint32_t* to) {
        src[k] = from;
        dst[k++] = to;
    }
};
// A read-back by one small kernel: the copies of `first`, then up to two runs of
// device words into pinned host memory (read it after a stream
// synchronisation).  A copy node costs a kernel as well and more of the host.
struct ReadBack {
    WordCopies first;
    const void* src[2] = {nullptr, nullptr};
    void* host[2] = {nullptr, nullptr};
    int words[2] = {0, 0};  // 32-bit words
};
void read_back(const ReadBack& r, hipStream_t s);

// In-place exclusive scans of k <= kMaxScanSet arrays of one length n, each
// array's total to its entry n (every array holds n + 1 entries), in two
// launches for all of them; tmp holds tmp_words uint32 (separate scans
// where that is too few or n exceeds 4096 * 4096).
constexpr int kMaxScanSet = 8;
struct ScanSet {
    uint32_t* a[kMaxScanSet];
};
void exclusive_scan_set_u32(const ScanSet& set, int k, int64_t n, uint32_t* tmp, size_t tmp_words,
                            hipStream_t s, const uint32_t* n_dev = nullptr);

// Stable LSD radix sort of (key, value) pairs by the low `bits` bits of the
// key.  Returns true when the result is in (keys_b, vals_b), false when it is
// in (keys_a, vals_a).  `hist` must hold radix_hist_words(n) uint32 and `tmp`
// scan_tmp_words(radix_hist_words(n)).
size_t radix_hist_words(int64_t n);
// The same with the key's significant bits in device memory (*bits_dev <=
// max_bits, 8-bit digits; passes beyond the bits do nothing): the result is
// always in (keys_a, vals_a).
template <typename K>
void radix_sort_pairs_dev(K* keys_a, uint32_t* vals_a, K* keys_b, uint32_t* vals_b, int64_t n,
                          int max_bits, const int* bits_dev, uint32_t* hist, uint32_t* tmp,
                          hipStream_t s);
template <typename K>
bool radix_sort_pairs(K* keys_a, uint32_t* vals_a, K* keys_b, uint32_t* vals_b, int64_t n,
                      int bits, uint32_t* hist, uint32_t* tmp, hipStream_t s);
// radix_sort_pairs (n > 1, bits > 0, pairs of row index i -> row i) that
// also moves the rows: row i of pts (D values) lands where its pair does,
// in soa (D planes of stride ld); rows_a and rows_b (n * D values each; b
// only with three passes or more) hold the rows between passes.  Reading
// each tile's rows where it lies replaces a gather of random rows after
// the sort.  Instantiated for rows of 4 or 8 bytes (float, D <= 2; double,
// D = 1): wider rows would take LDS that the sort's occupancy needs.
template <typename K, typename T, int D>
bool radix_sort_pairs_rows(K* keys_a, uint32_t* vals_a, K* keys_b, uint32_t* vals_b, int64_t n,
                           int bits, uint32_t* hist, uint32_t* tmp, const T* pts, T* rows_a,
                           T* rows_b, T* soa, int64_t ld, hipStream_t s);
int radix_pass_count(int bits);  // passes of radix_sort_pairs over `bits` key bits
template <typename T, int D>
constexpr bool sort_moves_rows() {
    return (std::is_same<T, float>::value && D <= 2) || (std::is_same<T, double>::value && D == 1);
}

// Grid geometry of the eps-grid, computed on the host from the min/max of
// the data exactly as the reference does (spatial_index.h:124-142).
struct Geometry {
    int d = 0;
    uint64_t cells[kMaxDims] = {};   // cells per input dimension
    int swapped[kMaxDims] = {};      // dimension order, fewest cells first
    uint64_t stride[kMaxDims] = {};  // stride of swapped dimension k
    uint64_t ncell[kMaxDims] = {};   // cells of swapped dimension k
    uint64_t total = 1;              // product of cells (wrapping)
    bool overflow = false;           // product exceeded 2^64
    int key_bits = 0;                // bits of the largest cell id
};

// Device-side parameter blocks.
struct CellParams {
    int d;
    int swapped[kMaxDims];
    uint64_t stride[kMaxDims];
    uint64_t ncell[kMaxDims];
};

// Everything a kernel needs to know about one clustering job (one point
// cloud with its own eps and minPts).  A plain call is a batch of one job.
// Jobs are laid out back to back: rows [row_begin, row_end) of the
// concatenated input, cell keys [key_base, key_base + total cells).  After
// the sort by key, a job's sorted positions are again [row_begin, row_end).
template <typename T>
struct JobParams {
    CellParams cp;
    uint64_t key_base = 0;
    int64_t row_begin = 0;
    int64_t row_end = 0;
    T minv[kMaxDims] = {};  // per-dimension minimum: the grid origin
    T eps2{};               // EPS2 converted to T
    float rcp_f = 0.0f;     // 1/eps in float (float and integer data)
    double rcp_d = 0.0;     // 1/eps in double (double data)
    uint32_t min_pts = 0;
};

// last j < n with at_or_below(j), ascending and true for j = 0, by the whole wave:
// 64 places per step (two dependent loads for 4096 jobs, a halving search 12)
template <typename Fn>
__device__ __forceinline__ int32_t wave_last(int32_t n, Fn&& at_or_below) {
    const int32_t lane = static_cast<int32_t>(threadIdx.x & 63);
    int32_t lo = 0, len = n;
    while (len > 1) {
        const int32_t step = (len + 63) / 64;
        const int32_t i = lane * step;
        const int32_t k = __popcll(__ballot(i < len && at_or_below(lo + i))) - 1;
        lo += k * step;
        len = min(step, len - k * step);
    }
    return __builtin_amdgcn_readfirstlane(lo);
}

// job index of a row (rows sorted by job): last j with row_begin <= row; every
// lane of the wave, one row
template <typename T>
__device__ __forceinline__ int32_t job_of_row(const JobParams<T>* __restrict__ jobs, int32_t njobs,
                                              int64_t row) {
    return wave_last(njobs, [&](int32_t j) { return jobs[j].row_begin <= row; });
}

// fn(job, row) for the rows [r0, r1) of a wave, 64 at a time on the lanes: rows
// of one job with a wave-uniform reference (scalar loads of the parameters),
// segments that span jobs with one per lane.  (Parameters read per lane: 4096
// clouds of 8k rows took 1.16 ms for the cell ids.)
template <typename T, typename Fn>
__device__ __forceinline__ void for_job_rows(const JobParams<T>* __restrict__ jobs, int32_t njobs,
                                             int64_t r0, int64_t r1, Fn&& fn) {
    auto scalar = [](int64_t v) {
        return static_cast<int64_t>(static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(
                   static_cast<int>(v & 0xffffffff)))) |
               (static_cast<int64_t>(
                    __builtin_amdgcn_readfirstlane(static_cast<int>(v >> 32)))
                << 32);
    };
    r0 = scalar(r0);
    r1 = scalar(r1);
    if (r0 >= r1) return;
    const int64_t lane = static_cast<int64_t>(threadIdx.x & 63);
    int32_t j = njobs == 1 ? 0 : job_of_row(jobs, njobs, r0);
    for (int64_t i0 = r0; i0 < r1; i0 += 64) {
        const int64_t last = (i0 + 64 < r1 ? i0 + 64 : r1) - 1;
        while (j + 1 < njobs && jobs[j].row_end <= i0) ++j;
        const int64_t i = i0 + lane;
        if (njobs == 1 || jobs[j].row_end > last) {
            if (i <= last) fn(jobs[j], i);
        } else if (i <= last) {
            int32_t k = j;
            while (k + 1 < njobs && jobs[k].row_end <= i) ++k;
            fn(jobs[k], i);
        }
    }
}

}  // namespace hpd
