// C-ABI of libhpdbscan_amd.so and the host orchestration of one clustering
// run.  The steps follow the reference's single-node path:
//
//   HPDBSCAN::HPDBSCAN / cluster<T>(T*, int, int)    hpdbscan.h:288-298, 475-486
//   SpatialIndex<T>::SpatialIndex                     spatial_index.h:528-628
//     min/max -> cells per dim -> dimension order -> cell ids -> sort
//   local_dbscan -> apply_rules -> recover_initial_order
//                                                     hpdbscan.h:372-448
#include <algorithm>
#include <cfloat>
#include <chrono>
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <limits>
#include <mutex>
#include <numeric>
#include <string>
#include <type_traits>
#include <vector>

#include "../../include/hpdbscan_capi.h"
#include "boxes.hpp"
#include "dbscan.hpp"
#include "grid.hpp"
#include "index.hpp"
#include "internal.hpp"
#include "small.hpp"

namespace hpd {

// --------------------------------------------------------------------------
// errors
// --------------------------------------------------------------------------
static thread_local std::string g_last_error;

void check_hip(hipError_t e, const char* what) {
    if (e != hipSuccess) {
        throw Error(e == hipErrorOutOfMemory ? HPD_ENOMEM : HPD_EDEVICE,
                    std::string(what) + ": " + hipGetErrorString(e));
    }
}

// --------------------------------------------------------------------------
// arena
// --------------------------------------------------------------------------
Arena::~Arena() {
    if (base_ && owned_) (void)hipFree(base_);
}

void Arena::reserve(size_t bytes) {
    used_ = 0;
    if (bytes <= cap_) return;
    if (!owned_)
        throw Error(HPD_EUNSUPPORTED, "the run needs " + std::to_string(bytes) +
                                          " bytes of device workspace here; " +
                                          std::to_string(cap_) + " are available");
    release();
    const size_t want = align_up(bytes + bytes / 8, size_t(1) << 20);
    void* p = nullptr;
    HPD_HIP(hipMalloc(&p, want));
    base_ = static_cast<char*>(p);
    cap_ = want;
}

void Arena::release() {
    if (!base_ || !owned_) return;
    HPD_HIP(hipFree(base_));
    base_ = nullptr;
    cap_ = used_ = 0;
}

void* Arena::take(size_t bytes) {
    const size_t b = align_up(bytes > 0 ? bytes : 1, 256);
    if (used_ + b > cap_) throw Error(HPD_ENOMEM, "internal: device workspace exhausted");
    void* p = base_ + used_;
    used_ += b;
    return p;
}

// --------------------------------------------------------------------------
// host-side arithmetic of the grid (reference build semantics)
// --------------------------------------------------------------------------

// The reference's -Ofast build runs with flush-to-zero and
// denormals-are-zero (crtfastmath.o); these helpers apply the same flushing
// to the few scalar steps evaluated on the host.
static inline float flushf(float x) { return std::fabs(x) < FLT_MIN ? 0.0f * x : x; }
static inline double flushd(double x) { return std::fabs(x) < DBL_MIN ? 0.0 * x : x; }

// float/double -> integer as x86-64 cvttss2si / cvttsd2si produce it
static inline int64_t f2i64_x86(double v) {
    if (!(v >= -9223372036854775808.0 && v < 9223372036854775808.0)) return INT64_MIN;
    return static_cast<int64_t>(v);
}
static inline int32_t f2i32_x86(double v) {
    if (!(v >= -2147483648.0 && v < 2147483648.0)) return INT32_MIN;
    return static_cast<int32_t>(v);
}
static inline uint64_t f2u64_x86(double v) {
    if (v < 9223372036854775808.0) return static_cast<uint64_t>(f2i64_x86(v));
    return static_cast<uint64_t>(f2i64_x86(v - 9223372036854775808.0)) ^ 0x8000000000000000ull;
}

template <typename T>
static float int_diff_f32_host(T x, T mn) {
    using P = decltype(x - mn);
    if constexpr (sizeof(T) < sizeof(int)) {
        return static_cast<float>(static_cast<int>(x) - static_cast<int>(mn));
    } else {
        using U = std::make_unsigned_t<P>;
        return static_cast<float>(static_cast<P>(static_cast<U>(x) - static_cast<U>(mn)));
    }
}

// cells per dimension, ceil((max - min) / eps) + 1 (spatial_index.h:124-131)
template <typename T>
static uint64_t cells_of(T mx, T mn, float rcp_f, double rcp_d) {
    if constexpr (std::is_same<T, float>::value) {
        const float v = flushf(flushf(flushf(mx) - flushf(mn)) * rcp_f);
        return f2u64_x86(static_cast<double>(std::ceil(v))) + 1;
    } else if constexpr (std::is_same<T, double>::value) {
        const double v = flushd(flushd(flushd(mx) - flushd(mn)) * rcp_d);
        return f2u64_x86(std::ceil(v)) + 1;
    } else {
        const float v = flushf(int_diff_f32_host<T>(mx, mn) * rcp_f);
        return f2u64_x86(static_cast<double>(std::ceil(v))) + 1;
    }
}

// EPS2 = (float)(eps * eps) (hpdbscan.h:53), converted to T when passed to
// region_query (spatial_index.h:739)
template <typename T>
static T eps2_as(float eps) {
    const float f = flushf(flushf(eps) * flushf(eps));
    if constexpr (std::is_same<T, float>::value) {
        return f;
    } else if constexpr (std::is_same<T, double>::value) {
        return static_cast<double>(f);
    } else if constexpr (std::is_same<T, uint64_t>::value) {
        return f2u64_x86(static_cast<double>(f));
    } else if constexpr (std::is_same<T, int64_t>::value) {
        return f2i64_x86(static_cast<double>(f));
    } else if constexpr (std::is_same<T, uint32_t>::value) {
        return static_cast<uint32_t>(f2i64_x86(static_cast<double>(f)));
    } else {
        return static_cast<T>(f2i32_x86(static_cast<double>(f)));
    }
}

template <typename T>
static Geometry make_geometry(const T* mn, const T* mx, int d, float eps, float* rcp_f_out,
                              double* rcp_d_out) {
    Geometry g;
    g.d = d;
    const float rcp_f = flushf(1.0f / flushf(eps));
    const double rcp_d = flushd(1.0 / flushd(static_cast<double>(eps)));
    *rcp_f_out = rcp_f;
    *rcp_d_out = rcp_d;
    uint64_t total = 1;
    bool overflow = false;
    for (int j = 0; j < d; ++j) {
        g.cells[j] = cells_of<T>(mx[j], mn[j], rcp_f, rcp_d);
        uint64_t t;
        if (__builtin_mul_overflow(total, g.cells[j], &t)) overflow = true;
        total *= g.cells[j];
    }
    g.total = total;
    g.overflow = overflow;
    // dimension order: the reference's own call, std::sort ascending by cell
    // count (spatial_index.h:135-139)
    size_t sw[kMaxDims];
    std::iota(sw, sw + d, size_t(0));
    std::sort(sw, sw + d, [&](size_t a, size_t b) { return g.cells[a] < g.cells[b]; });
    uint64_t acc = 1;
    for (int k = 0; k < d; ++k) {
        g.swapped[k] = static_cast<int>(sw[k]);
        g.stride[k] = acc;
        g.ncell[k] = g.cells[g.swapped[k]];
        acc *= g.ncell[k];
    }
    const uint64_t maxkey = total - 1;
    g.key_bits = maxkey == 0 ? 0 : 64 - __builtin_clzll(maxkey);
    return g;
}

// Host array of n elements: inline storage up to N (a single job needs no
// heap allocation), the heap beyond.
template <typename U, size_t N>
class HostArray {
public:
    explicit HostArray(size_t n) : n_(n) {
        if (n > N) heap_.resize(n);
        p_ = n > N ? heap_.data() : inl_;
        for (size_t i = 0; i < n; ++i) p_[i] = U{};
    }
    HostArray(const HostArray&) = delete;
    HostArray& operator=(const HostArray&) = delete;
    U* data() { return p_; }
    U& operator[](size_t i) { return p_[i]; }
    size_t size() const { return n_; }

private:
    size_t n_;
    U inl_[N];
    std::vector<U> heap_;
    U* p_;
};

// --------------------------------------------------------------------------
// context
// --------------------------------------------------------------------------
constexpr int kHostMinMax = 64, kHostWords = 128;  // of Context::host_scratch

struct Context {
    int device = 0;
    hipStream_t stream = nullptr;
    Arena main;
    Arena aux;
    Arena io;  // input rows and labels of the host-memory entry point
    // the arenas a run takes its workspace from: main / aux, or the static
    // scratch (hpd_cluster_device_noalloc)
    Arena* main_use = &main;
    Arena* aux_use = &aux;
    int border_rule = HPD_BORDER_MIN_CLUSTER;
    // hpd_context_set_work_split: kept for its getter
    int32_t sparse_max = 8;
    bool sparse_core = false;
    // sub-boxes per cell and dimension (hpd_context_set_box_split; 0: 2 up
    // to 3-D, 3 above, which keeps every sub-box's diagonal below eps)
    int32_t box_split = 0;
    uint64_t open_pair_limit = 0;  // 0: one entry per row
    // entries of a list of put-off work of a run of n rows
    unsigned long long put_off_cap(uint64_t n) const {
        return open_pair_limit > 0 && open_pair_limit < n ? open_pair_limit : n;
    }
    bool timing = false;
    bool count_tests = false;  // hpd_context_set_timing level 2
    hpd_run_stats stats{};
    // pinned: small results and read-backs; from kHostMinMax on the min / max of a
    // run of one job (2 * kMaxDims values, then the non-finite flag)
    uint64_t* host_scratch = nullptr;
    std::vector<hipEvent_t> events;
    // hpd_context_set_graph: floating-point runs go through the static
    // pipeline, captured in a hipGraph and replayed while the shape stays
    bool graph = false;
    struct GraphEntry {
        hipGraphExec_t exec = nullptr;
        int dtype = -1, d = 0, border_rule = -1, box_split = -1;
        bool count_tests = false;
        int64_t n = 0;
        const void* data = nullptr;
        const void* labels = nullptr;
        const void* arena_main = nullptr;
        const void* arena_aux = nullptr;
        std::vector<int64_t> offsets;
    } graph_entry;
    uint64_t graph_launches = 0, graph_captures = 0, graph_fallbacks = 0;
};

struct DeviceGuard {
    int prev = -1;
    explicit DeviceGuard(int dev) {
        HPD_HIP(hipGetDevice(&prev));
        if (prev != dev) HPD_HIP(hipSetDevice(dev));
    }
    ~DeviceGuard() {
        int cur = -1;
        if (hipGetDevice(&cur) == hipSuccess && prev >= 0 && cur != prev) (void)hipSetDevice(prev);
    }
};

// Named points of a run at which HIP events are recorded on the run's
// stream (when timing is on).
enum Mark : int {
    M_START,
    M_GRID,        // min/max and cell ids done
    M_SORT,        // both sorts and the gather done
    M_INDEX,       // cells, neighbour rows, boxes done
    M_CORE0,       // the core count kernel starts (after the full boxes' flags)
    M_CORE,        // core flags done
    M_HOOK0,       // box union: hook forest starts
    M_HOOK1,       // box union: hook forest and its roots done
    M_JOIN1,       // box union: union kernel done
    M_UNION,       // clusters of all cores known
    M_BORDER0,     // core labels written, border pass starts
    M_LABELS,      // all labels written
    M_COUNT
};

class PhaseTimer {
public:
    PhaseTimer(Context& c, hipStream_t s) : ctx_(c), s_(s) {}
    void mark(Mark m) {
        hipEvent_t e = event(m);
        if (e) HPD_HIP(hipEventRecord(e, s_));
    }
    // the event of mark m for the caller to record (null when timing is off)
    hipEvent_t event(Mark m) {
        if (!ctx_.timing) return nullptr;
        while (ctx_.events.size() < M_COUNT) {
            hipEvent_t e;
            HPD_HIP(hipEventCreate(&e));
            ctx_.events.push_back(e);
        }
        seen_[m] = true;
        return ctx_.events[m];
    }
    // milliseconds between two recorded marks (after a stream sync); 0 if
    // either was not recorded in this run
    double ms(Mark i, Mark j) const {
        if (!ctx_.timing || !seen_[i] || !seen_[j]) return 0.0;
        float v = 0.0f;
        HPD_HIP(hipEventElapsedTime(&v, ctx_.events[i], ctx_.events[j]));
        return static_cast<double>(v);
    }

private:
    Context& ctx_;
    hipStream_t s_;
    bool seen_[M_COUNT] = {};
};

// --------------------------------------------------------------------------
// one clustering run
// --------------------------------------------------------------------------
// Neighbour rows of one run are indexed with 32-bit offsets (signed in the
// kernels' loops).
constexpr uint64_t kMaxNeighborRows = 0x7fffffffull;
constexpr int kWaveRows = 64;  // rows of a work item
// 64-bit device words of a run: statistics (0-7), 32-bit counters (8-15, of
// which 15 counts the union's heavy entries), put-off walks of the core count
// (16) and of the border pass (17, 18)
constexpr int kStatWords = 24;

static void check_neighbor_rows(uint64_t total) {
    if (total > kMaxNeighborRows)
        throw Error(HPD_EUNSUPPORTED,
                    "the run has " + std::to_string(total) +
                        " neighbour rows (non-empty rows of 3 adjacent cells, summed over the "
                        "occupied cells); at most 2^31-1 are supported");
}

// sub-boxes per cell and dimension of a run of dimension d
static int split_of(const Context& c, int d) { return c.box_split > 0 ? c.box_split : box_split(d); }

static inline int bits_for(uint64_t max_value) {
    return max_value == 0 ? 0 : 64 - __builtin_clzll(max_value);
}

// device bytes of the job table and the min/max pass of a run
template <typename T, int D>
static size_t table_bytes(int64_t n, int64_t njobs) {
    const size_t nn = static_cast<size_t>(n), nj = static_cast<size_t>(njobs);
    const size_t mm_blocks = nn / static_cast<size_t>(minmax_rows_per_block(n)) + nj + 1;
    return sizeof(T) * 2 * D * (mm_blocks + nj) + 4 * (mm_blocks + nj + 2) + 64 +
           sizeof(JobParams<T>) * nj + 8 * 256;
}

// most neighbour rows of n rows: 3^(D-1) per cell
template <int D>
constexpr int64_t range_bound(int64_t n) {
    int64_t r = n;
    for (int j = 1; j < D; ++j) r *= 3;
    return r;
}

// worst-case device workspace of one run with n rows
template <typename T, int D>
static size_t workspace_bytes(int64_t n, int64_t njobs, bool one_thread) {
    const size_t nn = static_cast<size_t>(n);
    const size_t L = align_up(nn, 16);
    const size_t hist_words = radix_hist_words(n);
    const size_t tmp_words = scan_tmp_words(static_cast<int64_t>(std::max(hist_words, 2 * nn + 2)));
    size_t b = 0;
    b += 2 * 8 * nn + 2 * 4 * nn;              // keys / values of the sort
    b += 4 * hist_words + 4 * tmp_words;       // radix histogram, scan scratch
    b += sizeof(T) * L * D;                    // coordinates in slot order
    b += 4 * (2 * nn + 2);                     // run flags + scan
    b += 8 * nn + 4 * 4 * (nn + 1);            // ucell, ustart, nranges, nchunks, core chunks
    b += L + 3 * 4 * L + 3 * 4 * nn;           // core, parent, rsnap, rootslot, cmin/cmax/rcenter
    b += 8 * nn + 2 * 4 * nn + 3 * 4 * (nn + 1) + 5 * 4 * nn + nn;  // scratch64, positions, box tables
    b += 2 * D * 8 * nn;                       // box bounding boxes
    b += gather_part_bytes(n, D, static_cast<int>(sizeof(T)));  // their per-block shares
    if (sort_moves_rows<T, D>()) b += 2 * sizeof(T) * D * nn;   // rows between sort passes
    b += table_bytes<T, D>(n, njobs) + 4 * nn;  // job table, min/max, job of every cell
    if (one_thread) b += 8 * nn + 4 * nn + nn + 4;  // ambiguous rows, f, involved, flag
    b += 8 * kStatWords;                       // statistics, counters
    b += 54 * 256 + 64 * 1024;                 // alignment
    return b;
}

template <typename T, int D, typename K>
static void run_keyed(Context& ctx, const T* pts, int64_t n, JobParams<T>* jobs,
                      const JobParams<T>* host_jobs, int32_t njobs, int key_bits, uint64_t key_total, bool use_boxes,
                      int64_t* labels, hipStream_t s, PhaseTimer& tm) {
    // (known false for integer rows: their box kernels are not compiled)
    const bool boxes = std::is_floating_point<T>::value && use_boxes;
    Arena& A = *ctx.main_use;
    Arena& X = *ctx.aux_use;
    const size_t nn = static_cast<size_t>(n);
    const int64_t ld = (n + 15) & ~int64_t(15);  // rows are read in aligned batches of <= 16
    const size_t L = static_cast<size_t>(ld);
    // each key buffer is followed by its value buffer, so that the pair the
    // sort leaves free is one block (the dense cell table's room)
    K* keys_a = A.take_n<K>(nn);
    uint32_t* vals_a = A.take_n<uint32_t>(nn);
    K* keys_b = A.take_n<K>(nn);
    uint32_t* vals_b = A.take_n<uint32_t>(nn);
    const size_t hist_words = radix_hist_words(n);
    uint32_t* hist = A.take_n<uint32_t>(hist_words);
    const size_t tmp_words = scan_tmp_words(static_cast<int64_t>(std::max(hist_words, 2 * nn + 2)));
    uint32_t* tmp = A.take_n<uint32_t>(tmp_words);
    T* soa = A.take_n<T>(L * D);
    uint32_t* flags = A.take_n<uint32_t>(2 * nn + 2);
    K* ucell = A.take_n<K>(nn);
    int32_t* ustart = A.take_n<int32_t>(nn + 1);
    uint32_t* nranges = A.take_n<uint32_t>(nn + 1);
    uint32_t* nchunks = A.take_n<uint32_t>(nn + 1);
    uint8_t* core = A.take_n<uint8_t>(L);
    int32_t* parent = A.take_n<int32_t>(L);
    int32_t* rsnap = A.take_n<int32_t>(L);
    int32_t* rootslot = A.take_n<int32_t>(L);
    int32_t* cmin = A.take_n<int32_t>(nn);
    int32_t* cmax = A.take_n<int32_t>(nn);
    int32_t* rcenter = A.take_n<int32_t>(nn);
    int32_t* job_of_cell = A.take_n<int32_t>(nn);
    unsigned long long* dstats = A.take_n<unsigned long long>(kStatWords);
    // 0 m, 1 ranges, 2 items, 3 boxes, 5 loose, 6 chunks to count, 7 non-core
    // rows, 8 boxes with cores, 9 roots, 10 boxes near several trees, 11 and 12 large boxes, 13 full-row table
    uint32_t* counters = reinterpret_cast<uint32_t*>(dstats + 8);
    // the job table and the zeroed counters
    if (njobs == 1) {
        launch_put_job<T>(host_jobs[0], jobs, dstats, kStatWords * sizeof(unsigned long long), s);
    } else {
        HPD_HIP(hipMemcpyAsync(jobs, host_jobs, sizeof(JobParams<T>) * njobs,
                               hipMemcpyHostToDevice, s));
        HPD_HIP(hipMemsetAsync(dstats, 0, kStatWords * sizeof(unsigned long long), s));
    }
    uint32_t* hc = reinterpret_cast<uint32_t*>(ctx.host_scratch);

    // cell ids (spatial_index.h:144-165), offset by the job's key base; in
    // box mode followed by the row's sub-box digit, so that one stable sort
    // orders the rows by cell, then sub-box, then input row
    const int sub_k = split_of(ctx, D);
    const int sub_bits = boxes ? box_sub_bits(D, sub_k) : 0;
    launch_cell_ids<T, D, K>(pts, n, jobs, njobs, sub_k, sub_bits, keys_a, vals_a, s);
    tm.mark(M_GRID);

    // stable sort (spatial_index.h:167-216): slot -> input row; jobs stay
    // contiguous and in order because their key ranges are.  Rows of up to
    // 16 bytes travel with their pairs into soa (a gather of random rows
    // afterwards reads a whole cache line per row).
    const int sort_bits = key_bits + sub_bits;
    const bool rows_sorted = sort_moves_rows<T, D>() && n > 1 && sort_bits > 0;
    bool in_b = false;
    if (rows_sorted) {
        const int passes = radix_pass_count(sort_bits);
        T* rows_a = passes > 1 ? A.take_n<T>(nn * D) : nullptr;
        T* rows_b = passes > 2 ? A.take_n<T>(nn * D) : nullptr;
        in_b = radix_sort_pairs_rows<K, T, D>(keys_a, vals_a, keys_b, vals_b, n, sort_bits, hist,
                                              tmp, pts, rows_a, rows_b, soa, ld, s);
    } else {
        in_b = radix_sort_pairs<K>(keys_a, vals_a, keys_b, vals_b, n, sort_bits, hist, tmp, s);
    }
    K* keys = in_b ? keys_b : keys_a;
    uint32_t* inrow_of_slot = in_b ? vals_b : vals_a;
    K* keys_free = in_b ? keys_a : keys_b;
    uint32_t* vals_free = in_b ? vals_a : vals_b;

    // occupied cells (spatial_index.h:167-182); their order and the order of
    // input rows inside them are the reference's sorted order (box mode:
    // from the boxes, below)
    if (!boxes) launch_cells<K>(keys, n, sub_bits, flags, tmp, ucell, ustart, &counters[0], s);

    // box mode: slots are rows sorted by cell, sub-box, input row; the
    // reference's sorted positions are only materialised where needed
    uint32_t* pos_of_slot = nullptr;
    int32_t *box_of_slot = nullptr, *bstart = nullptr, *bcell = nullptr, *cbox = nullptr;
    int32_t *bmincore = nullptr, *bparent = nullptr, *compmin = nullptr, *bcluster = nullptr;
    uint8_t* btight = nullptr;
    void* bbox = nullptr;
    int32_t* ctab = nullptr;
    uint64_t* scratch64 = nullptr;  // n words: open-pair lists, position sort
    if (boxes) {
        scratch64 = A.take_n<uint64_t>(nn);
        pos_of_slot = A.take_n<uint32_t>(nn);
        box_of_slot = A.take_n<int32_t>(nn);
        bstart = A.take_n<int32_t>(nn + 1);
        bcell = A.take_n<int32_t>(nn);
        cbox = A.take_n<int32_t>(nn + 1);
        bmincore = A.take_n<int32_t>(nn);
        bparent = A.take_n<int32_t>(nn);
        compmin = A.take_n<int32_t>(nn);
        bcluster = A.take_n<int32_t>(nn);
        btight = A.take_n<uint8_t>(nn);
        bbox = A.take(2 * D * sizeof(T) * nn);
        void* bpart = A.take(gather_part_bytes(n, D, static_cast<int>(sizeof(T))));
        // a dense table of every cell id in the sort's spare key buffer, when
        // the grid is small enough (the neighbour rows then read the table
        // instead of searching the occupied cells)
        const size_t free_pair = align_up(nn * sizeof(K), 256) + nn * sizeof(uint32_t);
        if (key_total > 0 && key_total <= free_pair / sizeof(int32_t)) {
            ctab = reinterpret_cast<int32_t*>(keys_free);  // keys_free and vals_free
            fill_i32(ctab, -1, static_cast<int64_t>(key_total), s);
        }
        launch_box_table<K>(keys, n, sub_bits, flags, box_of_slot, bstart, bcell, ucell, ustart,
                            cbox, ctab, &counters[3], &counters[0], s);
        launch_gather_boxes<T, D>(rows_sorted ? nullptr : pts, n, inrow_of_slot, soa, ld,
                                  box_of_slot, bstart, bbox, bpart, s);
    } else if (!rows_sorted) {
        launch_gather_soa<T, D>(pts, n, inrow_of_slot, soa, ld, s);
    }
    // one read-back for the occupied cells and the boxes
    ReadBack cells;
    cells.src[0] = counters;
    cells.host[0] = hc;
    cells.words[0] = 4;
    read_back(cells, s);
    HPD_HIP(hipStreamSynchronize(s));
    const int32_t m = static_cast<int32_t>(hc[0]);
    const int32_t nbox = boxes ? static_cast<int32_t>(hc[3]) : 0;
    tm.mark(M_SORT);

    // neighbour ranges (spatial_index.h:682-737)
    uint8_t* cell_core = boxes ? A.take_n<uint8_t>(nn) : nullptr;
    // the count pass keeps the rows it finds in scratch64 (idle until the
    // core count) when every cell's 3^(D-1) rows fit, and the fill copies them
    constexpr int32_t max_rows = static_cast<int32_t>(range_bound<D>(1));
    int2* stash = scratch64 && !neighbor_rows_wide(m, max_rows) &&
                          static_cast<uint64_t>(m) * static_cast<uint64_t>(max_rows) <= nn
                      ? reinterpret_cast<int2*>(scratch64)
                      : nullptr;
    // up to 27 rows per cell (D <= 4): the copy puts the nearest rows first
    const bool by_class = stash && D <= 4;
    launch_neighbor_count<K, T>(ucell, ustart, host_count(m), jobs, njobs, job_of_cell, nranges,
                                cell_core, &dstats[0], &dstats[4], stash, max_rows, rcenter,
                                by_class, s, ctab);
    // the per-cell counts, scanned together (totals at entry m); box mode
    // has no use for the 64-row chunks of every cell unless the union runs on
    // rows or the one-thread border rule meets an ambiguous row
    if (!boxes) launch_chunk_counts(ustart, host_count(m), nchunks, s);
    ScanSet counts{};
    int ncounts = 0;
    counts.a[ncounts++] = nranges;
    if (!boxes) counts.a[ncounts++] = nchunks;
    exclusive_scan_set_u32(counts, ncounts, m, tmp, tmp_words, s);
    if (boxes) {
        // the box flags (their loose count decides the union) before the
        // read-back below
        BoxArgs<T> bt;
        bt.nbox = nbox;
        bt.bstart = bstart;
        bt.bcell = bcell;
        bt.bbox = bbox;
        bt.jobs = jobs;
        bt.job_of_cell = job_of_cell;
        launch_box_tight<T, D>(bt, cell_core, btight, &counters[5], heavy_walk_rows(), &counters[11],
                               s);
    }
    // the scans' totals into the counters (one launch), then one read-back
    // of the 64-bit row total (dstats[4]) and the counters (dstats + 8)
    ReadBack totals;
    totals.first.add(&nranges[m], &counters[1]);
    if (!boxes) totals.first.add(&nchunks[m], &counters[2]);
    unsigned long long* hs_rows = reinterpret_cast<unsigned long long*>(ctx.host_scratch) + 12;
    totals.src[0] = &dstats[4];
    totals.host[0] = hs_rows;
    totals.words[0] = 24;
    read_back(totals, s);
    HPD_HIP(hipStreamSynchronize(s));
    hc = reinterpret_cast<uint32_t*>(hs_rows + 4);  // the counters as read back
    // the scan of nranges and every range index are 32-bit: check the
    // 64-bit total first
    check_neighbor_rows(*hs_rows);
    const uint32_t total_ranges = hc[1];
    // every box of two or more rows is tight: the union runs on boxes
    const bool all_tight = boxes && hc[5] == 0;
    const bool one_thread = ctx.border_rule == HPD_BORDER_ONE_THREAD;
    // the row-level tables: slot and cell ranges of the neighbour rows and the
    // chunks of every cell (at most one per cell and one per 64 rows)
    const bool row_tables = !all_tight || one_thread;
    const size_t max_items =
        boxes ? static_cast<size_t>(m) + nn / kWaveRows + 1 : static_cast<size_t>(hc[2]);

    const size_t range_bytes = align_up(static_cast<size_t>(total_ranges) * sizeof(int2), 256);
    // (the cell ranges take the box ranges' place when they are made)
    X.reserve((boxes ? range_bytes : 0) + (row_tables ? (boxes ? 1 : 2) * range_bytes : 0) +
              (row_tables ? align_up(max_items * sizeof(int2), 256) : 0) + 2048);
    int2* rboxes = boxes ? X.take_n<int2>(total_ranges) : nullptr;
    int2* ranges = row_tables ? X.take_n<int2>(total_ranges) : nullptr;
    int2* rcells = !row_tables ? nullptr : boxes ? rboxes : X.take_n<int2>(total_ranges);
    int2* items = row_tables ? X.take_n<int2>(max_items) : nullptr;
    if (boxes && stash)
        launch_neighbor_copy(stash, max_rows, m, nranges, cbox, rboxes, rcenter, by_class, s);
    else if (boxes)
        launch_neighbor_fill<K, T>(ucell, ustart, host_count(m), jobs, job_of_cell, nranges,
                                   nullptr, rboxes, rcenter, max_rows, s, ctab, cbox);
    else
        launch_neighbor_fill<K, T>(ucell, ustart, host_count(m), jobs, job_of_cell, nranges,
                                   ranges, rcells, rcenter, max_rows, s);
    if (!boxes)
        launch_work_items(ustart, host_count(m), nchunks, host_count(static_cast<int64_t>(hc[2])),
                          items, s);

    DbscanArgs<T> a;
    a.soa = soa;
    a.n = n;
    a.ld = ld;
    a.items = items;
    a.nitems = boxes ? 0 : static_cast<int32_t>(hc[2]);
    a.ustart = ustart;
    a.roff = nranges;
    a.ranges = ranges;
    a.rcells = rcells;
    a.rcenter = rcenter;
    a.m = m;
    a.jobs = jobs;
    a.njobs = njobs;
    a.job_of_cell = job_of_cell;
    a.pos_of_slot = nullptr;  // slots are positions unless boxes reorder them
    a.inrow = inrow_of_slot;

    BoxArgs<T> ba;
    bool box_union = false;
    if (boxes) {
        ba.soa = soa;
        ba.ld = ld;
        ba.nbox = nbox;
        ba.bstart = bstart;
        ba.bcell = bcell;
        ba.cbox = cbox;
        ba.bbox = bbox;
        ba.jobs = jobs;
        ba.njobs = njobs;
        ba.nrows = n;
        ba.job_of_cell = job_of_cell;
        ba.rcenter = rcenter;
        a.box_of_slot = box_of_slot;
        a.btight = btight;
        a.cbox = cbox;
        a.bstart = bstart;
        a.bcell = bcell;
        a.bbox = bbox;
        a.rboxes = rboxes;
        a.bmincore = bmincore;
        // both row lists in scratch64, before and after the union
        a.crows = reinterpret_cast<int2*>(scratch64);
        a.ncrows_dev = &counters[6];
        a.brows = reinterpret_cast<int2*>(scratch64);
        a.nbrows_dev = &counters[7];
        if (hc[11] > 0) {  // boxes of millions of rows: their walks in parts
            a.heavy = reinterpret_cast<int2*>(flags);
            a.nheavy = &dstats[16];
            a.heavy_cap = ctx.put_off_cap(nn);
            a.slot_a = parent;  // free before and after the union
            a.slot_b = rsnap;
            a.late = cmin;
            a.nlate = reinterpret_cast<unsigned int*>(&dstats[18]);
        }
    }
    // box mode: the row-level tables when they turn out to be needed (the
    // neighbour rows ascending again, their own-row index with them); the box
    // ranges are gone after it, no kernel on boxes follows
    auto fill_row_tables = [&] {
        launch_chunk_counts(ustart, host_count(m), nchunks, s);
        exclusive_scan_u32(nchunks, nchunks, m, tmp, &nchunks[m], s);
        uint32_t* h = reinterpret_cast<uint32_t*>(ctx.host_scratch) + 64;
        HPD_HIP(hipMemcpyAsync(h, &nchunks[m], sizeof(uint32_t), hipMemcpyDeviceToHost, s));
        HPD_HIP(hipStreamSynchronize(s));
        a.nitems = static_cast<int32_t>(*h);
        launch_work_items(ustart, host_count(m), nchunks, host_count(a.nitems), items, s);
        launch_neighbor_fill<K, T>(ucell, ustart, host_count(m), jobs, job_of_cell, nranges,
                                   ranges, rcells, rcenter, max_rows, s);
    };
    tm.mark(M_INDEX);

    launch_core<T, D>(a, core, ctx.count_tests ? &dstats[7] : nullptr, s, tm.event(M_CORE0));
    tm.mark(M_CORE);

    // box lists of the union (box mode leaves the slot-level parent free)
    // (the lists' lengths stay on the device: boxes with cores, and the
    // roots of each join round)
    int32_t* blist = parent;
    box_union = all_tight;
    if (box_union) {
        // compmin holds the forest's roots until the clusters are known; the
        // smallest key of every cluster lies in flags, between the put-off
        // walks of the core count and those of the border pass
        unsigned long long* cluster_keys = reinterpret_cast<unsigned long long*>(flags);
        tm.mark(M_HOOK0);
        launch_list_boxes(host_count(nbox), bmincore, blist, &counters[8], bparent, cluster_keys, s);
        launch_box_hook<T, D>(ba, nranges, rboxes, bmincore, core, blist, &counters[8], bparent, s);
        // (the slot-level union's rsnap is free in box mode: the roots)
        launch_box_roots(host_count(nbox), bmincore, bparent, compmin, rsnap, &counters[9], s);
        launch_box_root_join<T, D>(ba, nranges, rboxes, compmin, core, rsnap, &counters[9], bparent,
                                   s);
        launch_box_roots(host_count(nbox), bmincore, bparent, compmin, nullptr, nullptr, s);
        tm.mark(M_HOOK1);
        // pairs with a large box go through a list in scratch64
        const unsigned long long cap = ctx.put_off_cap(nn);
        launch_box_union<T, D>(ba, nranges, rboxes, compmin, core, blist, &counters[8],
                               host_count(m), rsnap, &counters[10], box_of_slot,
                               reinterpret_cast<int2*>(scratch64), &dstats[15], cap, bparent,
                               &dstats[5], hc[12] > 0, s);
        tm.mark(M_JOIN1);
        launch_box_clusters(host_count(nbox), bmincore, bcell, cbox, bstart, inrow_of_slot, ustart,
                            bparent, cluster_keys, compmin,
                            bcluster, s);
    } else {
        if (boxes) {
            // a loose box: the slot-level union needs the sorted positions
            // and the row-level tables
            fill_row_tables();
            launch_positions(n, m, box_of_slot, bcell, inrow_of_slot,
                             reinterpret_cast<uint32_t*>(keys), vals_free,
                             reinterpret_cast<uint32_t*>(keys_free),
                             reinterpret_cast<uint32_t*>(scratch64), hist, tmp, pos_of_slot, s);
            a.pos_of_slot = pos_of_slot;
        }
        if (!compmin) compmin = A.take_n<int32_t>(nn);
        launch_union_points<T, D>(a, core, parent, rsnap, cmin, cmax, compmin, s);
    }
    tm.mark(M_UNION);
    int2* amb = one_thread ? A.take_n<int2>(nn) : nullptr;
    // box mode reads rootslot only under the one-thread border rule; without
    // it the rows of full boxes are labelled in input order, through a table
    // indexed by cell key in the sort's spare key buffer when the keys fit
    // (launched only when every key fits the table; *full_ok stays 0 else)
    const bool full_rows = box_union && !one_thread &&
                           key_total <= (nn * sizeof(K) / sizeof(int32_t)) >> sub_bits;
    unsigned int* full_ok = full_rows ? &counters[13] : nullptr;
    if (full_rows)
        launch_label_full_rows<T, D, K>(pts, a, sub_k, sub_bits, keys, host_count(nbox),
                                        bcluster, reinterpret_cast<int32_t*>(keys_free),
                                        static_cast<int64_t>(nn * sizeof(K) / 4), labels,
                                        full_ok, s);
    launch_label_cores<T>(a, core, box_union ? bcluster : nullptr, parent, compmin,
                          box_union && !one_thread ? nullptr : rootslot, cmin, cmax, labels,
                          &dstats[1], s, full_ok);
    tm.mark(M_BORDER0);
    a.nheavy = &dstats[17];
    launch_border<T, D>(a, core, box_union ? bcluster : nullptr, rootslot, cmin, cmax, labels,
                        &dstats[2], amb, s);

    unsigned long long* hs = reinterpret_cast<unsigned long long*>(ctx.host_scratch);
    ReadBack sums;
    sums.src[0] = dstats;
    sums.host[0] = hs;
    sums.words[0] = 16;
    read_back(sums, s);
    HPD_HIP(hipStreamSynchronize(s));
    if (box_union) ctx.stats.open_box_pairs = hs[5];
    ctx.stats.core_tests = hs[7];
    if (one_thread && hs[3] > 0) {
        // the reference's choice at one thread for the border rows next to
        // two or more clusters (hpdbscan.h:74-92)
        const int32_t namb = static_cast<int32_t>(hs[3]);
        if (box_union) fill_row_tables();
        if (boxes && !a.pos_of_slot) {  // the relaxation compares sorted positions
            launch_positions(n, m, box_of_slot, bcell, inrow_of_slot,
                             reinterpret_cast<uint32_t*>(keys), vals_free,
                             reinterpret_cast<uint32_t*>(keys_free),
                             reinterpret_cast<uint32_t*>(scratch64), hist, tmp, pos_of_slot, s);
            a.pos_of_slot = pos_of_slot;
        }
        int32_t* f = A.take_n<int32_t>(nn);
        uint8_t* involved = A.take_n<uint8_t>(nn);
        unsigned int* changed = A.take_n<unsigned int>(1);
        HPD_HIP(hipMemsetAsync(involved, 0, nn, s));
        launch_one_thread_mark<T, D>(a, core, rootslot, amb, namb, involved, f, s);
        // sweep k leaves every core whose best decreasing path has at most
        // k steps final, so sweep n + 1 at the latest changes nothing.  A
        // sweep that changes nothing is a fixed point; the host reads the
        // flag of the last sweep of a batch, and the batches double (up to
        // 64 sweeps), so a long chain costs few read-backs
        int64_t sweeps = 0;
        for (int batch = 1;; batch = std::min(2 * batch, 64)) {
            if (sweeps > n + 1) throw Error(HPD_EDEVICE, "border relaxation did not converge");
            for (int i = 0; i < batch; ++i) {
                if (i == batch - 1) HPD_HIP(hipMemsetAsync(changed, 0, sizeof(unsigned int), s));
                launch_one_thread_relax<T, D>(a, core, rootslot, involved, f, changed, s);
            }
            sweeps += batch;
            HPD_HIP(hipMemcpyAsync(hc + 32, changed, sizeof(unsigned int), hipMemcpyDeviceToHost, s));
            HPD_HIP(hipStreamSynchronize(s));
            if (hc[32] == 0) break;
        }
        launch_one_thread_assign<T, D>(a, core, rootslot, amb, namb, f, labels, s);
    }
    tm.mark(M_LABELS);
    // labels are complete on return; the timing events are read next
    if (ctx.timing || (one_thread && hs[3] > 0)) HPD_HIP(hipStreamSynchronize(s));
    ctx.stats.sum_candidates = hs[0];
    ctx.stats.core_points = hs[1];
    ctx.stats.noise_points = hs[2];
    ctx.stats.ambiguous_borders = hs[3];
    ctx.stats.occupied_cells = static_cast<uint64_t>(m);
    ctx.stats.neighbor_rows = total_ranges;
    ctx.stats.boxes = static_cast<uint64_t>(nbox);
    ctx.stats.box_union = box_union ? 1 : 0;
}

// --------------------------------------------------------------------------
// small inputs
// --------------------------------------------------------------------------
// Waits for a small run's result and takes its statistics; false when it
// refused the input (the general path then runs it, or reports why not), or
// left ambiguous border rows to the one-thread rule.
static bool read_small(Context& ctx, hipStream_t s) {
    HPD_HIP(hipStreamSynchronize(s));
    const SmallResult* r = reinterpret_cast<const SmallResult*>(ctx.host_scratch);
    if (r->nonfinite || r->overflow || r->unfit ||
        (r->ambiguous > 0 && ctx.border_rule == HPD_BORDER_ONE_THREAD))
        return false;
    ctx.stats.total_cells = r->total_cells;
    ctx.stats.key_bits = bits_for(r->total_cells - 1);
    ctx.stats.sum_candidates = r->sum_candidates;
    ctx.stats.core_points = r->cores;
    ctx.stats.noise_points = r->noise;
    ctx.stats.ambiguous_borders = r->ambiguous;
    ctx.stats.occupied_cells = r->cells;
    ctx.stats.neighbor_rows = r->neighbor_rows;
    ctx.stats.boxes = r->boxes;
    return true;
}

template <typename T, int D>
static size_t small_call_bytes(int64_t n) {
    return small_workspace_bytes<T, D>(n) + align_up(sizeof(SmallResult), 256);
}

// One job of few rows through the all-pairs kernels (small.hip).
template <typename T, int D>
static bool run_small(Context& ctx, const T* pts, int64_t n, float eps, uint64_t min_pts,
                      int64_t* labels, hipStream_t s) {
    Arena& A = *ctx.main_use;
    A.reserve(small_call_bytes<T, D>(n));
    SmallResult* result = A.take_n<SmallResult>(1);
    void* work = A.take(small_workspace_bytes<T, D>(n));
    JobParams<T> jp{};
    jp.row_end = n;
    jp.min_pts = static_cast<uint32_t>(std::min<uint64_t>(min_pts, 0xffffffffull));
    jp.eps2 = eps2_as<T>(eps);
    jp.rcp_f = flushf(1.0f / flushf(eps));
    jp.rcp_d = flushd(1.0 / flushd(static_cast<double>(eps)));
    const int sub_k = split_of(ctx, D);
    launch_small<T, D>(pts, n, jp, nullptr, sub_k, box_sub_bits(D, sub_k), work, result,
                       reinterpret_cast<SmallResult*>(ctx.host_scratch), labels, s);
    return read_small(ctx, s);
}

// --------------------------------------------------------------------------
// the static pipeline (hpd_context_set_graph)
// --------------------------------------------------------------------------
// The same kernels as run_keyed, with every table sized by its worst case
// from n, the number of jobs and D, and every count that run_keyed reads back
// to size the next step left in device memory (a Count with a device
// address, the kernels reading it; wave kernels walk their items from a
// bounded grid).  The grid of every job is computed on the device
// (launch_geometry) and the radix passes beyond its key bits do nothing, so
// no host read-back happens between the first kernel and the last: the
// sequence can be captured in a hipGraph and replayed.  Conditions on which
// run_keyed branches become flags read after the run; any of them hands the
// run to the plain pipeline: non-finite input, grids beyond 64 key bits,
// loose boxes.  Box mode only
// (floating-point data), smallest-cluster border rule.

// Device words the static pipeline keeps its counts in.
enum StaticSlot : int {
    SS_M = 0,          // occupied cells
    SS_RANGES = 1,     // neighbour rows
    SS_NBOX = 3,       // boxes
    SS_LOOSE = 5,      // boxes of two or more rows that are not tight
    SS_CROWS = 6,      // rows to count
    SS_BROWS = 7,      // non-core rows
    SS_NLIST = 8,      // boxes with cores
    SS_JOIN = 9,       // roots of the hook forest
    SS_MIXED = 10,     // boxes of cells next to several trees
    SS_LARGE = 11,     // and 12 (boxes above a size: not used here)
    SS_NONFINITE = 14, // non-finite coordinates
    SS_GRID = 15,      // grid beyond 64 key bits
    SS_BITS = 16,      // key bits + sub-box bits
    SS_ROWTAB = 17,    // the row-order label table holds every key
    SS_WORDS = 32
};

template <typename T, int D>
static size_t static_aux_bytes(int64_t n) {
    return align_up(static_cast<size_t>(range_bound<D>(n)) * sizeof(int2), 256) +
           4096;
}

template <typename T, int D>
static size_t static_main_bytes(int64_t n, int32_t njobs) {
    size_t b = workspace_bytes<T, D>(n, njobs, false);
    if (njobs == 1 && n <= small_rows(D))  // all pairs compared: a bit per pair
        b = std::max(b, table_bytes<T, D>(n, 1) + small_workspace_bytes<T, D>(n));
    return b + sizeof(uint64_t) * static_cast<size_t>(njobs) + SS_WORDS * 4 + sizeof(SmallResult) +
           64 * 1024 + 8 * 256;
}

// The body of a static run on stream s: every launch of the run, nothing
// else (no read-back, no synchronisation, no memset), in the workspace the
// caller reserved and started taking from; jobs / bfirst_dev hold the
// host-made job table (row ranges, eps2, minPts, reciprocals) and min/max
// blocks.  sc (SS_WORDS words) and dstats (kStatWords words) end up
// holding the counts read afterwards.
template <typename T, int D>
static void static_body(Context& ctx, const T* pts, int64_t n, JobParams<T>* jobs,
                        const int32_t* bfirst_dev, int32_t njobs, int32_t nblocks, int64_t* labels,
                        uint32_t* sc, unsigned long long* dstats, SmallResult* small,
                        hipStream_t s) {
    using K = uint64_t;
    Arena& A = ctx.main;
    Arena& X = ctx.aux;
    X.reset();
    if (njobs == 1 && n <= small_rows(D)) {
        const int parts = split_of(ctx, D);
        void* work = A.take(small_workspace_bytes<T, D>(n));
        launch_small<T, D>(pts, n, JobParams<T>{}, jobs, parts, box_sub_bits(D, parts), work, small,
                           reinterpret_cast<SmallResult*>(ctx.host_scratch), labels, s);
        return;
    }
    const size_t nn = static_cast<size_t>(n);
    const int64_t ld = (n + 15) & ~int64_t(15);
    const size_t L = static_cast<size_t>(ld);
    // zeroed by a kernel (no memset in a graph)
    fill_i32(reinterpret_cast<int32_t*>(sc), 0, SS_WORDS, s);
    fill_i32(reinterpret_cast<int32_t*>(dstats), 0, 2 * kStatWords, s);

    // min / max, then every job's grid on the device
    T* part = A.take_n<T>(static_cast<size_t>(nblocks) * 2 * D + 1);
    T* mm = A.take_n<T>(static_cast<size_t>(njobs) * 2 * D + 16);
    uint64_t* jcells = A.take_n<uint64_t>(static_cast<size_t>(njobs));
    unsigned long long* total_cells = dstats + 6;
    int* bad_part = A.take_n<int>(static_cast<size_t>(nblocks) + 1);
    launch_minmax<T, D>(pts, 0, n, jobs, njobs, bfirst_dev, nblocks, minmax_rows_per_block(n), part,
                        bad_part, mm, reinterpret_cast<int*>(&sc[SS_NONFINITE]), s);
    const int sub_k = split_of(ctx, D);
    const int sub_bits = box_sub_bits(D, sub_k);
    launch_geometry<T, D>(jobs, njobs, mm, sub_bits, jcells, reinterpret_cast<int*>(&sc[SS_GRID]),
                          reinterpret_cast<int*>(&sc[SS_BITS]), total_cells, s);

    K* keys_a = A.take_n<K>(nn);
    K* keys_b = A.take_n<K>(nn);
    uint32_t* vals_a = A.take_n<uint32_t>(nn);
    uint32_t* vals_b = A.take_n<uint32_t>(nn);
    const size_t hist_words = radix_hist_words(n);
    uint32_t* hist = A.take_n<uint32_t>(hist_words);
    const size_t tmp_words = scan_tmp_words(static_cast<int64_t>(std::max(hist_words, 2 * nn + 2)));
    uint32_t* tmp = A.take_n<uint32_t>(tmp_words);
    T* soa = A.take_n<T>(L * D);
    uint32_t* flags = A.take_n<uint32_t>(2 * nn + 2);
    K* ucell = A.take_n<K>(nn);
    int32_t* ustart = A.take_n<int32_t>(nn + 1);
    uint32_t* nranges = A.take_n<uint32_t>(nn + 1);
    uint32_t* nchunks = A.take_n<uint32_t>(nn + 1);
    uint8_t* core = A.take_n<uint8_t>(L);
    int32_t* parent = A.take_n<int32_t>(L);
    int32_t* roots = A.take_n<int32_t>(L);  // (rsnap of the slot-level union)
    int32_t* rootslot = A.take_n<int32_t>(L);
    int32_t* cmin = A.take_n<int32_t>(nn);
    int32_t* cmax = A.take_n<int32_t>(nn);
    int32_t* rcenter = A.take_n<int32_t>(nn);
    int32_t* job_of_cell = A.take_n<int32_t>(nn);
    uint64_t* scratch64 = A.take_n<uint64_t>(nn);
    (void)A.take_n<uint32_t>(nn);  // sorted positions (loose boxes only)
    int32_t* box_of_slot = A.take_n<int32_t>(nn);
    int32_t* bstart = A.take_n<int32_t>(nn + 1);
    int32_t* bcell = A.take_n<int32_t>(nn);
    int32_t* cbox = A.take_n<int32_t>(nn + 1);
    int32_t* bmincore = A.take_n<int32_t>(nn);
    int32_t* bparent = A.take_n<int32_t>(nn);
    int32_t* compmin = A.take_n<int32_t>(nn);
    int32_t* bcluster = A.take_n<int32_t>(nn);
    uint8_t* btight = A.take_n<uint8_t>(nn);
    void* bbox = A.take(2 * D * sizeof(T) * nn);
    void* bpart = A.take(gather_part_bytes(n, D, static_cast<int>(sizeof(T))));
    uint8_t* cell_core = A.take_n<uint8_t>(nn);

    // cell ids and the sort (passes past the key's bits do nothing)
    launch_cell_ids<T, D, K>(pts, n, jobs, njobs, sub_k, sub_bits, keys_a, vals_a, s);
    radix_sort_pairs_dev<K>(keys_a, vals_a, keys_b, vals_b, n, 64,
                            reinterpret_cast<const int*>(&sc[SS_BITS]), hist, tmp, s);
    K* keys = keys_a;
    uint32_t* inrow_of_slot = vals_a;
    launch_box_table<K>(keys, n, sub_bits, flags, box_of_slot, bstart, bcell, ucell, ustart, cbox,
                        nullptr, &sc[SS_NBOX], &sc[SS_M], s);
    launch_gather_boxes<T, D>(pts, n, inrow_of_slot, soa, ld, box_of_slot, bstart, bbox, bpart, s);

    // neighbour rows and work lists, counted and laid out on the device
    const Count M{n, &sc[SS_M]};
    const Count NB{n, &sc[SS_NBOX]};
    launch_neighbor_count<K, T>(ucell, ustart, M, jobs, njobs, job_of_cell, nranges, cell_core,
                                &dstats[0], &dstats[4], nullptr,
                                static_cast<int32_t>(range_bound<D>(1)), rcenter, false, s);
    exclusive_scan_u32_dev(nranges, nranges, M, tmp, s);
    copy_at_count(nranges, &sc[SS_M], &sc[SS_RANGES], s);
    const int64_t R = range_bound<D>(n);
    int2* rboxes = X.take_n<int2>(static_cast<size_t>(R));
    launch_neighbor_fill<K, T>(ucell, ustart, M, jobs, job_of_cell, nranges, nullptr, rboxes,
                               rcenter, static_cast<int32_t>(range_bound<D>(1)), s, nullptr, cbox);

    BoxArgs<T> ba;
    ba.soa = soa;
    ba.ld = ld;
    ba.nbox = static_cast<int32_t>(n);
    ba.nbox_dev = &sc[SS_NBOX];
    ba.bstart = bstart;
    ba.bcell = bcell;
    ba.cbox = cbox;
    ba.bbox = bbox;
    ba.jobs = jobs;
    ba.njobs = njobs;
    ba.nrows = n;
    ba.job_of_cell = job_of_cell;
    ba.rcenter = rcenter;
    launch_box_tight<T, D>(ba, cell_core, btight, &sc[SS_LOOSE], INT32_MAX, &sc[SS_LARGE], s);

    DbscanArgs<T> a;
    a.soa = soa;
    a.n = n;
    a.ld = ld;
    a.ustart = ustart;
    a.roff = nranges;
    a.rboxes = rboxes;
    a.rcenter = rcenter;
    a.m = static_cast<int32_t>(n);
    a.jobs = jobs;
    a.njobs = njobs;
    a.job_of_cell = job_of_cell;
    a.pos_of_slot = nullptr;
    a.inrow = inrow_of_slot;
    a.box_of_slot = box_of_slot;
    a.btight = btight;
    a.cbox = cbox;
    a.bstart = bstart;
    a.bcell = bcell;
    a.bbox = bbox;
    a.bmincore = bmincore;
    a.crows = reinterpret_cast<int2*>(scratch64);
    a.ncrows_dev = &sc[SS_CROWS];
    a.brows = reinterpret_cast<int2*>(scratch64);
    a.nbrows_dev = &sc[SS_BROWS];
    launch_core<T, D>(a, core, ctx.count_tests ? &dstats[7] : nullptr, s);

    // the box union (its result is discarded when a box is loose)
    unsigned long long* cluster_keys = reinterpret_cast<unsigned long long*>(flags);
    int32_t* blist = parent;
    launch_list_boxes(NB, bmincore, blist, &sc[SS_NLIST], bparent, cluster_keys, s);
    launch_box_hook<T, D>(ba, nranges, rboxes, bmincore, core, blist, &sc[SS_NLIST], bparent, s);
    launch_box_roots(NB, bmincore, bparent, compmin, roots, &sc[SS_JOIN], s);
    launch_box_root_join<T, D>(ba, nranges, rboxes, compmin, core, roots, &sc[SS_JOIN], bparent, s);
    launch_box_roots(NB, bmincore, bparent, compmin, nullptr, nullptr, s);
    launch_box_union<T, D>(ba, nranges, rboxes, compmin, core, blist, &sc[SS_NLIST], M, roots,
                           &sc[SS_MIXED], box_of_slot,
                           reinterpret_cast<int2*>(scratch64), &dstats[15],
                           static_cast<unsigned long long>(nn), bparent, &dstats[5], true, s);
    launch_box_clusters(NB, bmincore, bcell, cbox, bstart, inrow_of_slot, ustart, bparent,
                        cluster_keys, compmin, bcluster, s);

    // the rows of full boxes labelled in input order when the keys fit the
    // table (in the sort's spare key buffer), the other cores in slot order
    launch_label_full_rows<T, D, K>(pts, a, sub_k, sub_bits, keys, NB, bcluster,
                                    reinterpret_cast<int32_t*>(keys_b),
                                    static_cast<int64_t>(nn * sizeof(K) / 4), labels,
                                    &sc[SS_ROWTAB], s);
    launch_label_cores<T>(a, core, bcluster, parent, compmin, nullptr, cmin, cmax, labels,
                          &dstats[1], s, &sc[SS_ROWTAB]);
    launch_border<T, D>(a, core, bcluster, rootslot, cmin, cmax, labels, &dstats[2], nullptr, s);
    // counts, flags and statistics for the host
    ReadBack r;
    r.src[0] = sc;
    r.host[0] = ctx.host_scratch;
    r.words[0] = SS_WORDS;
    r.src[1] = dstats;
    r.host[1] = ctx.host_scratch + SS_WORDS / 2;
    r.words[1] = 16;
    read_back(r, s);
}

// Ends a stream capture if the body throws halfway.
struct CaptureGuard {
    hipStream_t s;
    bool open = true;
    ~CaptureGuard() {
        if (open) {
            hipGraph_t g = nullptr;
            if (hipStreamEndCapture(s, &g) == hipSuccess && g) (void)hipGraphDestroy(g);
        }
    }
};

// One batch through the static pipeline: replayed from the context's graph
// when the shape (dtype, D, rows, job offsets, buffers, options, workspace)
// matches the captured one, captured first otherwise.  Returns false when a
// flag hands the batch to the plain pipeline.
template <typename T, int D>
static bool run_static(Context& ctx, int dtype, const T* pts, int64_t n, const int64_t* offsets,
                       int32_t njobs, const float* eps, const uint64_t* min_pts, int64_t* labels,
                       hipStream_t s) {
    if (range_bound<D>(n) > 0x7fffffffll) return false;  // 32-bit range offsets
    ctx.main.reserve(static_main_bytes<T, D>(n, njobs));
    ctx.aux.reserve(static_aux_bytes<T, D>(n));
    Arena& A = ctx.main;
    A.reset();
    JobParams<T>* jobs_dev = A.take_n<JobParams<T>>(static_cast<size_t>(njobs));
    int32_t* bfirst_dev = A.take_n<int32_t>(static_cast<size_t>(njobs) + 1);
    uint32_t* sc = A.take_n<uint32_t>(SS_WORDS);
    unsigned long long* dstats = A.take_n<unsigned long long>(kStatWords);
    SmallResult* small = A.take_n<SmallResult>(1);

    // host-made part of the job table: row ranges, eps2, minPts, reciprocals
    HostArray<JobParams<T>, 1> hj(static_cast<size_t>(njobs));
    HostArray<int32_t, 2> bfirst(static_cast<size_t>(njobs) + 1);
    const int64_t rpb = minmax_rows_per_block(n);
    int32_t nblocks = 0;
    for (int32_t j = 0; j < njobs; ++j) {
        JobParams<T>& jp = hj[j];
        jp = JobParams<T>{};
        jp.row_begin = offsets[j];
        jp.row_end = offsets[j + 1];
        jp.min_pts = static_cast<uint32_t>(std::min<uint64_t>(min_pts[j], 0xffffffffull));
        jp.eps2 = eps2_as<T>(eps[j]);
        jp.rcp_f = flushf(1.0f / flushf(eps[j]));
        jp.rcp_d = flushd(1.0 / flushd(static_cast<double>(eps[j])));
        jp.cp.d = D;
        bfirst[j] = nblocks;
        nblocks += static_cast<int32_t>((offsets[j + 1] - offsets[j] + rpb - 1) / rpb);
    }
    bfirst[njobs] = nblocks;
    if (njobs == 1) {
        launch_put_job<T>(hj[0], jobs_dev, nullptr, 0, s);
    } else {
        HPD_HIP(hipMemcpyAsync(jobs_dev, hj.data(), sizeof(JobParams<T>) * njobs,
                               hipMemcpyHostToDevice, s));
        HPD_HIP(hipMemcpyAsync(bfirst_dev, bfirst.data(), sizeof(int32_t) * (njobs + 1),
                               hipMemcpyHostToDevice, s));
    }

    Context::GraphEntry& ge = ctx.graph_entry;
    const bool same = ge.exec && ge.dtype == dtype && ge.d == D && ge.n == n && ge.data == pts &&
                      ge.labels == labels && ge.arena_main == A.base() &&
                      ge.arena_aux == ctx.aux.base() && ge.border_rule == ctx.border_rule &&
                      ge.box_split == ctx.box_split && ge.count_tests == ctx.count_tests &&
                      ge.offsets.size() == static_cast<size_t>(njobs) + 1 &&
                      std::equal(ge.offsets.begin(), ge.offsets.end(), offsets);
    if (!same) {
        if (ge.exec) {
            (void)hipGraphExecDestroy(ge.exec);
            ge.exec = nullptr;
        }
        // captured on the context's stream, launched on s
        HPD_HIP(hipStreamSynchronize(ctx.stream));
        HPD_HIP(hipStreamBeginCapture(ctx.stream, hipStreamCaptureModeThreadLocal));
        CaptureGuard guard{ctx.stream};
        static_body<T, D>(ctx, pts, n, jobs_dev, bfirst_dev, njobs, nblocks, labels, sc, dstats,
                          small, ctx.stream);
        hipGraph_t g = nullptr;
        guard.open = false;
        HPD_HIP(hipStreamEndCapture(ctx.stream, &g));
        hipGraphExec_t exec = nullptr;
        const hipError_t e = hipGraphInstantiate(&exec, g, nullptr, nullptr, 0);
        (void)hipGraphDestroy(g);
        HPD_HIP(e);
        ge.exec = exec;
        ge.dtype = dtype;
        ge.d = D;
        ge.n = n;
        ge.data = pts;
        ge.labels = labels;
        ge.arena_main = A.base();
        ge.arena_aux = ctx.aux.base();
        ge.border_rule = ctx.border_rule;
        ge.box_split = ctx.box_split;
        ge.count_tests = ctx.count_tests;
        ge.offsets.assign(offsets, offsets + njobs + 1);
        ++ctx.graph_captures;
    }
    HPD_HIP(hipGraphLaunch(ge.exec, s));
    ++ctx.graph_launches;
    if (njobs == 1 && n <= small_rows(D)) {
        const bool taken = read_small(ctx, s);
        if (!taken) ++ctx.graph_fallbacks;
        return taken;
    }
    // the run's last kernel left the counts, flags and statistics here
    const uint32_t* hc = reinterpret_cast<const uint32_t*>(ctx.host_scratch);
    const unsigned long long* hs =
        reinterpret_cast<const unsigned long long*>(ctx.host_scratch) + SS_WORDS / 2;
    HPD_HIP(hipStreamSynchronize(s));
    const bool ok = hc[SS_NONFINITE] == 0 && hc[SS_GRID] == 0 && hc[SS_LOOSE] == 0 &&
                    hs[4] <= static_cast<unsigned long long>(range_bound<D>(n));
    if (!ok) {
        ++ctx.graph_fallbacks;
        return false;
    }
    ctx.stats.sum_candidates = hs[0];
    ctx.stats.core_points = hs[1];
    ctx.stats.noise_points = hs[2];
    ctx.stats.ambiguous_borders = hs[3];
    ctx.stats.open_box_pairs = hs[5];
    ctx.stats.core_tests = hs[7];
    ctx.stats.total_cells = hs[6];
    ctx.stats.key_bits = static_cast<int32_t>(hc[SS_BITS]) - box_sub_bits(D, split_of(ctx, D));
    ctx.stats.occupied_cells = hc[SS_M];
    ctx.stats.neighbor_rows = hc[SS_RANGES];
    ctx.stats.boxes = hc[SS_NBOX];
    ctx.stats.box_union = 1;
    return true;
}

// --------------------------------------------------------------------------
// integer rows as float rows
// --------------------------------------------------------------------------
// Integer rows whose arithmetic float reproduces exactly run as float rows,
// on boxes (200k lattice rows in 3-D: 5.1 ms by the row-level union of the
// integer path, whose wrapping distance is not monotone in general):
//   * coordinates and their spans at most 2^24: they are exact in float, and
//     so is every (x - min), whose float the reference's cell index takes;
//   * for any two rows that are candidates of each other, the squared
//     differences and their sum at most 2^24 (exact in float, in any order)
//     and at most the largest T (nothing wraps).  Candidates lie in the same
//     or in adjacent cells, so |x - y| / eps < 2 plus the rounding of the two
//     scaled values, each below span / eps <= 2^24 / eps.
// EPS2 is the integer path's (truncated) value.

// most |x - y| of candidates in a dimension of span `span` (both integers)
static double candidate_span(double span, float eps) {
    const double e = static_cast<double>(eps);
    const double b = (2.0 + span / e * (1.0 / (1 << 21))) * e * 1.00001 + 1.0;
    return std::min(span, std::floor(b));
}

// whether the sum of the squares of per-dimension spans stays exact
template <typename T>
static bool sum_exact(double sum) {
    return sum <= 16777216.0 && sum <= static_cast<double>(std::numeric_limits<T>::max());
}

template <typename T, int D>
static bool float_exact(const T* mn, const T* mx, float eps) {
    double sum = 0.0;
    for (int k = 0; k < D; ++k) {
        const double lo = static_cast<double>(mn[k]), hi = static_cast<double>(mx[k]);
        if (std::fabs(lo) > 16777216.0 || std::fabs(hi) > 16777216.0 || hi - lo > 16777216.0)
            return false;
        const double c = candidate_span(hi - lo, eps);
        sum += c * c;
    }
    return sum_exact<T>(sum);
}

// What float_exact needs whatever the data: whether it can hold for eps at
// all (the workspace for it is only taken then).  Spans below 2 eps can still
// pass it; such data has a few cells and stays on the integer path.
template <typename T, int D>
static bool float_possible(float eps) {
    return sum_exact<T>(static_cast<double>(D) * 4.0 * static_cast<double>(eps) *
                        static_cast<double>(eps));
}

// A batch of jobs: rows [offsets[j], offsets[j+1]) of `pts` form job j with
// its own eps[j] and min_pts[j].  A plain call is a batch of one.
// try_float: integer rows may run as float rows.
template <typename T, int D>
static void run_batch(Context& ctx, const T* pts, int64_t n, const int64_t* offsets,
                      int32_t njobs, const float* eps, const uint64_t* min_pts, int64_t* labels,
                      hipStream_t s, bool try_float = true) {
    if constexpr (std::is_floating_point<T>::value) {
        // the static pipeline, captured once per shape and replayed; it hands
        // the run back when one of its flags says so
        if (ctx.graph && ctx.border_rule == HPD_BORDER_MIN_CLUSTER && ctx.main_use == &ctx.main &&
            !ctx.timing &&
            run_static<T, D>(ctx, static_cast<int>(sizeof(T)), pts, n, offsets, njobs, eps, min_pts,
                             labels, s))
            return;
    }
    if constexpr (std::is_floating_point<T>::value) {
        // few rows: all pairs compared (the timing marks and the executed
        // tests are the general path's; a fixed workspace turns the marks off,
        // not the tests)
        if (njobs == 1 && n <= small_rows(D) && !ctx.timing && !ctx.count_tests &&
            run_small<T, D>(ctx, pts, n, eps[0], min_pts[0], labels, s))
            return;
    }
    PhaseTimer tm(ctx, s);
    tm.mark(M_START);
    Arena& A = *ctx.main_use;
    const bool one_thread = ctx.border_rule == HPD_BORDER_ONE_THREAD;
    bool as_float = false;  // integer rows: room for them as float rows
    if constexpr (std::is_integral<T>::value) {
        // (not in a fixed workspace, whose size the integer path's needs set)
        as_float = try_float && ctx.main_use == &ctx.main;
        for (int32_t j = 0; j < njobs && as_float; ++j) as_float = float_possible<T, D>(eps[j]);
        if (as_float) {
            try {
                A.reserve(workspace_bytes<float, D>(n, njobs, one_thread) +
                          table_bytes<T, D>(n, njobs) +
                          align_up(sizeof(float) * D * static_cast<size_t>(n), 256));
            } catch (const Error& e) {
                if (e.code != HPD_ENOMEM) throw;
                (void)hipGetLastError();
                as_float = false;
            }
        }
    }
    if (!as_float) A.reserve(workspace_bytes<T, D>(n, njobs, one_thread));

    // job table, first pass: row ranges and min/max blocks.  The host
    // vectors outlive every copy from them: the run ends with a stream sync.
    HostArray<JobParams<T>, 1> hj(static_cast<size_t>(njobs));
    HostArray<int32_t, 2> bfirst(static_cast<size_t>(njobs) + 1);
    const int64_t rpb = minmax_rows_per_block(n);
    int32_t nblocks = 0;
    for (int32_t j = 0; j < njobs; ++j) {
        hj[j] = JobParams<T>{};
        hj[j].row_begin = offsets[j];
        hj[j].row_end = offsets[j + 1];
        bfirst[j] = nblocks;
        nblocks += static_cast<int32_t>((offsets[j + 1] - offsets[j] + rpb - 1) / rpb);
    }
    bfirst[njobs] = nblocks;
    JobParams<T>* jobs_dev = A.take_n<JobParams<T>>(static_cast<size_t>(njobs));
    int32_t* bfirst_dev = A.take_n<int32_t>(static_cast<size_t>(njobs) + 1);
    T* part = A.take_n<T>(static_cast<size_t>(nblocks) * 2 * D + 1);
    T* mm = A.take_n<T>(static_cast<size_t>(njobs) * 2 * D + 16);
    int* nonfinite = reinterpret_cast<int*>(A.take_n<int>(4));
    int* bad_part = A.take_n<int>(static_cast<size_t>(nblocks) + 1);

    // min / max per job (spatial_index.h:99-122).  One job needs no table for
    // that, and its result goes to pinned memory by itself: 100k rows 362 -> 331 us
    // with the job table as a kernel argument and the read-backs as kernels.
    HostArray<T, 2 * D> hmm(static_cast<size_t>(njobs) * 2 * D);
    int hbad = 0;
    if (njobs == 1) {
        T* host_mm = reinterpret_cast<T*>(ctx.host_scratch + kHostMinMax);
        int* host_bad = reinterpret_cast<int*>(ctx.host_scratch + kHostMinMax + 2 * kMaxDims);
        launch_minmax<T, D>(pts, offsets[0], offsets[1], nullptr, 1, nullptr, nblocks, rpb, part,
                            bad_part, host_mm, host_bad, s);
        HPD_HIP(hipStreamSynchronize(s));
        std::memcpy(hmm.data(), host_mm, sizeof(T) * 2 * D);
        hbad = *host_bad;
    } else {
        HPD_HIP(hipMemcpyAsync(jobs_dev, hj.data(), sizeof(JobParams<T>) * njobs,
                               hipMemcpyHostToDevice, s));
        HPD_HIP(hipMemcpyAsync(bfirst_dev, bfirst.data(), sizeof(int32_t) * (njobs + 1),
                               hipMemcpyHostToDevice, s));
        HPD_HIP(hipMemsetAsync(nonfinite, 0, sizeof(int), s));
        launch_minmax<T, D>(pts, 0, n, jobs_dev, njobs, bfirst_dev, nblocks, rpb, part, bad_part,
                            mm, nonfinite, s);
        HPD_HIP(hipMemcpyAsync(hmm.data(), mm, sizeof(T) * njobs * 2 * D, hipMemcpyDeviceToHost,
                               s));
        HPD_HIP(hipMemcpyAsync(ctx.host_scratch, nonfinite, sizeof(int), hipMemcpyDeviceToHost,
                               s));
        HPD_HIP(hipStreamSynchronize(s));
        std::memcpy(&hbad, ctx.host_scratch, sizeof(int));
    }
    if (hbad) throw Error(HPD_EINVAL, "input contains NaN or infinite coordinates");

    // per-job grid (spatial_index.h:124-142) and key ranges
    uint64_t key_total = 0;
    for (int32_t j = 0; j < njobs; ++j) {
        JobParams<T>& jp = hj[j];
        jp.key_base = key_total;
        jp.min_pts = static_cast<uint32_t>(std::min<uint64_t>(min_pts[j], 0xffffffffull));
        jp.eps2 = eps2_as<T>(eps[j]);
        jp.cp.d = D;
        if (jp.row_end == jp.row_begin) continue;
        float rcp_f;
        double rcp_d;
        const T* mn = &hmm[static_cast<size_t>(j) * 2 * D];
        const Geometry g = make_geometry<T>(mn, mn + D, D, eps[j], &rcp_f, &rcp_d);
        if constexpr (std::is_integral<T>::value)
            as_float = as_float && float_exact<T, D>(mn, mn + D, eps[j]);
        if (g.overflow)
            throw Error(HPD_EUNSUPPORTED,
                        "the eps-grid has more than 2^64 cells (the reference's cell ids wrap)");
        jp.rcp_f = rcp_f;
        jp.rcp_d = rcp_d;
        for (int k = 0; k < D; ++k) {
            jp.minv[k] = mn[k];
            jp.cp.swapped[k] = g.swapped[k];
            jp.cp.stride[k] = g.stride[k];
            jp.cp.ncell[k] = g.ncell[k];
        }
        uint64_t t;
        if (__builtin_add_overflow(key_total, g.total, &t))
            throw Error(HPD_EUNSUPPORTED, "the jobs' grids have more than 2^64 cells together");
        key_total = t;
        if (njobs == 1) {
            ctx.stats.total_cells = g.total;
        }
    }
    if (njobs != 1) ctx.stats.total_cells = key_total;
    const int key_bits = bits_for(key_total > 0 ? key_total - 1 : 0);
    ctx.stats.key_bits = key_bits;

    // floating-point data (and integer data that float reproduces) runs on
    // sub-boxes (the sort key then carries the sub-box digit below the cell
    // id); other integer data, or a grid so large that the digit does not fit
    // beside the cell id, runs on cells
    const int split_bits = box_sub_bits(D, split_of(ctx, D));
    const bool boxes = (std::is_floating_point<T>::value || as_float) && key_bits + split_bits <= 64;
    const int sort_bits = key_bits + (boxes ? split_bits : 0);
    auto run = [&](auto* rows, auto* table, auto* host_table) {
        using R = std::remove_const_t<std::remove_pointer_t<decltype(rows)>>;
        if (sort_bits <= 32)
            run_keyed<R, D, uint32_t>(ctx, rows, n, table, host_table, njobs, key_bits, key_total, boxes,
                                      labels, s, tm);
        else
            run_keyed<R, D, uint64_t>(ctx, rows, n, table, host_table, njobs, key_bits, key_total, boxes,
                                      labels, s, tm);
    };
    if constexpr (std::is_integral<T>::value) {
        if (as_float && boxes) {
            HostArray<JobParams<float>, 1> hf(static_cast<size_t>(njobs));
            for (int32_t j = 0; j < njobs; ++j) {
                JobParams<float>& f = hf[j];
                f.cp = hj[j].cp;
                f.key_base = hj[j].key_base;
                f.row_begin = hj[j].row_begin;
                f.row_end = hj[j].row_end;
                for (int k = 0; k < D; ++k) f.minv[k] = static_cast<float>(hj[j].minv[k]);
                f.eps2 = static_cast<float>(hj[j].eps2);
                f.rcp_f = hj[j].rcp_f;
                f.rcp_d = hj[j].rcp_d;
                f.min_pts = hj[j].min_pts;
            }
            JobParams<float>* table = A.take_n<JobParams<float>>(static_cast<size_t>(njobs));
            float* rows = A.take_n<float>(static_cast<size_t>(n) * D);
            launch_to_float<T>(pts, n * D, rows, s);
            bool room = true;
            try {
                run(static_cast<const float*>(rows), table, hf.data());
            } catch (const Error& e) {
                if (e.code != HPD_ENOMEM) throw;
                (void)hipGetLastError();
                room = false;
            }
            if (!room) {
                // the float rows' workspace left none for the neighbour tables
                // (sized after the index, before any label is written): the
                // integer path, whose workspace is smaller
                A.release();
                return run_batch<T, D>(ctx, pts, n, offsets, njobs, eps, min_pts, labels, s, false);
            }
        }
    }
    if (std::is_floating_point<T>::value || !as_float || !boxes) {
        run(pts, jobs_dev, hj.data());
    }
    if (ctx.timing) {
        ctx.stats.ms_grid = tm.ms(M_START, M_GRID);
        ctx.stats.ms_sort = tm.ms(M_GRID, M_SORT);
        ctx.stats.ms_index = tm.ms(M_SORT, M_INDEX);
        ctx.stats.ms_core = tm.ms(M_INDEX, M_CORE);
        ctx.stats.ms_union = tm.ms(M_CORE, M_UNION);
        ctx.stats.ms_border = tm.ms(M_UNION, M_LABELS);
        ctx.stats.ms_total = tm.ms(M_START, M_LABELS);
        ctx.stats.ms_hook_kernel = tm.ms(M_HOOK0, M_HOOK1);
        ctx.stats.ms_union_kernel = tm.ms(M_HOOK1, M_JOIN1);
        ctx.stats.ms_border_kernel = tm.ms(M_BORDER0, M_LABELS);
        ctx.stats.ms_core_kernel = tm.ms(M_CORE0, M_CORE);
    }
}

template <typename T>
static void run_typed(Context& ctx, const T* pts, int64_t n, int d, const int64_t* offsets,
                      int32_t njobs, const float* eps, const uint64_t* min_pts, int64_t* labels,
                      hipStream_t s) {
    switch (d) {
        case 1: return run_batch<T, 1>(ctx, pts, n, offsets, njobs, eps, min_pts, labels, s);
        case 2: return run_batch<T, 2>(ctx, pts, n, offsets, njobs, eps, min_pts, labels, s);
        case 3: return run_batch<T, 3>(ctx, pts, n, offsets, njobs, eps, min_pts, labels, s);
        case 4: return run_batch<T, 4>(ctx, pts, n, offsets, njobs, eps, min_pts, labels, s);
        case 5: return run_batch<T, 5>(ctx, pts, n, offsets, njobs, eps, min_pts, labels, s);
        case 6: return run_batch<T, 6>(ctx, pts, n, offsets, njobs, eps, min_pts, labels, s);
        case 7: return run_batch<T, 7>(ctx, pts, n, offsets, njobs, eps, min_pts, labels, s);
        case 8: return run_batch<T, 8>(ctx, pts, n, offsets, njobs, eps, min_pts, labels, s);
        default:
            throw Error(HPD_EUNSUPPORTED, "dimensions above " + std::to_string(kMaxDims) +
                                              " are not supported by this build");
    }
}

static size_t dtype_size(int dt) {
    switch (dt) {
        case HPD_DTYPE_F32: return 4;
        case HPD_DTYPE_F64: return 8;
        case HPD_DTYPE_I8: case HPD_DTYPE_U8: return 1;
        case HPD_DTYPE_I16: case HPD_DTYPE_U16: return 2;
        case HPD_DTYPE_I32: case HPD_DTYPE_U32: return 4;
        case HPD_DTYPE_I64: case HPD_DTYPE_U64: return 8;
        default: return 0;
    }
}

static void run_any(Context& ctx, int dt, const void* pts, int64_t n, int d,
                    const int64_t* offsets, int32_t njobs, const float* eps,
                    const uint64_t* min_pts, int64_t* labels, hipStream_t s) {
#define HPD_RUN_CASE(CODE, T)                                                                \
    case CODE:                                                                               \
        return run_typed(ctx, static_cast<const T*>(pts), n, d, offsets, njobs, eps, min_pts, \
                         labels, s);
    switch (dt) {
        HPD_RUN_CASE(HPD_DTYPE_F32, float)
        HPD_RUN_CASE(HPD_DTYPE_F64, double)
        HPD_RUN_CASE(HPD_DTYPE_I8, int8_t)
        HPD_RUN_CASE(HPD_DTYPE_I16, int16_t)
        HPD_RUN_CASE(HPD_DTYPE_I32, int32_t)
        HPD_RUN_CASE(HPD_DTYPE_I64, int64_t)
        HPD_RUN_CASE(HPD_DTYPE_U8, uint8_t)
        HPD_RUN_CASE(HPD_DTYPE_U16, uint16_t)
        HPD_RUN_CASE(HPD_DTYPE_U32, uint32_t)
        HPD_RUN_CASE(HPD_DTYPE_U64, uint64_t)
        default: throw Error(HPD_EINVAL, "unknown dtype code " + std::to_string(dt));
    }
#undef HPD_RUN_CASE
}

// workspace of a plain call (one job) of any dtype and dimension: the general
// path's, and that of the all-pairs kernels where they are tried first
template <typename T, int D>
static size_t workspace_call(int64_t n, bool one_thread) {
    size_t b = workspace_bytes<T, D>(n, 1, one_thread);
    if constexpr (std::is_floating_point<T>::value)
        if (n <= small_rows(D)) b = std::max(b, small_call_bytes<T, D>(n));
    return b;
}

template <typename T>
static size_t workspace_typed(int64_t n, int d, bool one_thread) {
    switch (d) {
        case 1: return workspace_call<T, 1>(n, one_thread);
        case 2: return workspace_call<T, 2>(n, one_thread);
        case 3: return workspace_call<T, 3>(n, one_thread);
        case 4: return workspace_call<T, 4>(n, one_thread);
        case 5: return workspace_call<T, 5>(n, one_thread);
        case 6: return workspace_call<T, 6>(n, one_thread);
        case 7: return workspace_call<T, 7>(n, one_thread);
        case 8: return workspace_call<T, 8>(n, one_thread);
        default:
            throw Error(HPD_EUNSUPPORTED, "dimensions above " + std::to_string(kMaxDims) +
                                              " are not supported by this build");
    }
}

static size_t workspace_any(int dt, int64_t n, int d, bool one_thread) {
    switch (dt) {
        case HPD_DTYPE_F32: return workspace_typed<float>(n, d, one_thread);
        case HPD_DTYPE_F64: return workspace_typed<double>(n, d, one_thread);
        case HPD_DTYPE_I8: return workspace_typed<int8_t>(n, d, one_thread);
        case HPD_DTYPE_I16: return workspace_typed<int16_t>(n, d, one_thread);
        case HPD_DTYPE_I32: return workspace_typed<int32_t>(n, d, one_thread);
        case HPD_DTYPE_I64: return workspace_typed<int64_t>(n, d, one_thread);
        case HPD_DTYPE_U8: return workspace_typed<uint8_t>(n, d, one_thread);
        case HPD_DTYPE_U16: return workspace_typed<uint16_t>(n, d, one_thread);
        case HPD_DTYPE_U32: return workspace_typed<uint32_t>(n, d, one_thread);
        case HPD_DTYPE_U64: return workspace_typed<uint64_t>(n, d, one_thread);
        default: throw Error(HPD_EINVAL, "unknown dtype code " + std::to_string(dt));
    }
}

// --------------------------------------------------------------------------
// static scratch of hpd_cluster_device_noalloc
// --------------------------------------------------------------------------
// Every workspace buffer of a run of hpd_cluster_device_noalloc lives in
// this array (one copy per device, held until the process ends).  Host code
// never passes its name to a kernel: the name is a host-side stand-in; the
// device address comes from hipGetSymbolAddress, looked up once per device
// when a context is created on it (with that device current).
constexpr size_t kScratchBytes = size_t(128) << 20;
static __device__ __align__(256) unsigned char scratch[kScratchBytes];

constexpr int kMaxDevices = 64;
static std::mutex g_scratch_mu;
static void* g_scratch_ptr[kMaxDevices] = {};

static void init_scratch_for_current_device(int device) {
    if (device < 0 || device >= kMaxDevices)
        throw Error(HPD_EUNSUPPORTED, "device index above " + std::to_string(kMaxDevices - 1));
    std::lock_guard<std::mutex> lock(g_scratch_mu);
    if (g_scratch_ptr[device]) return;
    void* ptr = nullptr;
    HPD_HIP(hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch)));
    if (!ptr) throw Error(HPD_EDEVICE, "hipGetSymbolAddress returned a null scratch address");
    g_scratch_ptr[device] = ptr;
}

static void* scratch_of(int device) {
    std::lock_guard<std::mutex> lock(g_scratch_mu);
    return device >= 0 && device < kMaxDevices ? g_scratch_ptr[device] : nullptr;
}

// Points a context's runs at fixed arenas and turns its timing off (event
// creation) for the duration of one call.
class FixedWorkspace {
public:
    FixedWorkspace(Context& c, void* base, size_t main_bytes, size_t total_bytes)
        : c_(c), timing_(c.timing) {
        main_.attach(base, main_bytes);
        aux_.attach(static_cast<char*>(base) + main_bytes, total_bytes - main_bytes);
        c.main_use = &main_;
        c.aux_use = &aux_;
        c.timing = false;
    }
    ~FixedWorkspace() {
        c_.main_use = &c_.main;
        c_.aux_use = &c_.aux;
        c_.timing = timing_;
    }
    FixedWorkspace(const FixedWorkspace&) = delete;
    FixedWorkspace& operator=(const FixedWorkspace&) = delete;

private:
    Context& c_;
    bool timing_;
    Arena main_, aux_;
};

static void validate(const Context* ctx, int dt, const void* data, int64_t n, int32_t d, float eps,
                     const void* labels) {
    if (!ctx) throw Error(HPD_EINVAL, "context is NULL");
    // hpdbscan.h:295-297 (NaN is rejected as well)
    if (!(eps > 0.0f)) throw Error(HPD_EINVAL, "epsilon needs to be positive");
    if (dtype_size(dt) == 0) throw Error(HPD_EINVAL, "unknown dtype code " + std::to_string(dt));
    if (n < 0) throw Error(HPD_EINVAL, "the number of rows must not be negative");
    if (n > 0x7fffffffll) throw Error(HPD_EINVAL, "at most 2^31-1 rows (the reference takes an int)");
    if (d < 1) throw Error(HPD_EINVAL, "the number of dimensions must be positive");
    if (n > 0 && (!data || !labels)) throw Error(HPD_EINVAL, "data and labels must not be NULL");
}

}  // namespace hpd

using hpd::Context;
using hpd::Error;

struct hpd_context {
    Context impl;
};

template <typename F>
static int guarded(F&& f) {
    try {
        f();
        hpd::g_last_error.clear();
        return HPD_OK;
    } catch (const Error& e) {
        hpd::g_last_error = e.what();
        return e.code;
    } catch (const std::bad_alloc&) {
        hpd::g_last_error = "host allocation failed";
        return HPD_ENOMEM;
    } catch (const std::exception& e) {
        hpd::g_last_error = e.what();
        return HPD_EDEVICE;
    }
}

extern "C" {

const char* hpd_last_error(void) { return hpd::g_last_error.c_str(); }

const char* hpd_version(void) { return "hpdbscan-amd 0.1.0 (gfx950)"; }

int hpd_device_count(void) {
    int n = 0;
    if (hipGetDeviceCount(&n) != hipSuccess) return 0;
    return n;
}

int hpd_context_create(int device, hpd_context** out) {
    return guarded([&] {
        if (!out) throw Error(HPD_EINVAL, "out is NULL");
        *out = nullptr;
        int count = 0;
        if (hipGetDeviceCount(&count) != hipSuccess || count == 0)
            throw Error(HPD_EDEVICE, "no HIP device is available");
        if (device < 0 || device >= count)
            throw Error(HPD_EINVAL, "device index " + std::to_string(device) + " out of range");
        auto* c = new hpd_context();
        try {
            c->impl.device = device;
            hpd::DeviceGuard g(device);
            hpd::init_scratch_for_current_device(device);
            HPD_HIP(hipStreamCreateWithFlags(&c->impl.stream, hipStreamNonBlocking));
            void* hs = nullptr;
            HPD_HIP(hipHostMalloc(&hs, hpd::kHostWords * sizeof(uint64_t), hipHostMallocDefault));
            c->impl.host_scratch = static_cast<uint64_t*>(hs);
        } catch (...) {
            if (c->impl.stream) (void)hipStreamDestroy(c->impl.stream);
            delete c;
            throw;
        }
        *out = c;
    });
}

int hpd_context_destroy(hpd_context* ctx) {
    return guarded([&] {
        if (!ctx) return;
        {
            hpd::DeviceGuard g(ctx->impl.device);
            if (ctx->impl.stream) (void)hipStreamSynchronize(ctx->impl.stream);
            if (ctx->impl.graph_entry.exec) (void)hipGraphExecDestroy(ctx->impl.graph_entry.exec);
            for (auto e : ctx->impl.events) (void)hipEventDestroy(e);
            if (ctx->impl.host_scratch) (void)hipHostFree(ctx->impl.host_scratch);
            if (ctx->impl.stream) (void)hipStreamDestroy(ctx->impl.stream);
        }
        delete ctx;
    });
}

int hpd_context_set_border_rule(hpd_context* ctx, int rule) {
    return guarded([&] {
        if (!ctx) throw Error(HPD_EINVAL, "context is NULL");
        if (rule != HPD_BORDER_MIN_CLUSTER && rule != HPD_BORDER_ONE_THREAD)
            throw Error(HPD_EINVAL, "unknown border rule");
        ctx->impl.border_rule = rule;
    });
}

int hpd_context_set_timing(hpd_context* ctx, int enabled) {
    return guarded([&] {
        if (!ctx) throw Error(HPD_EINVAL, "context is NULL");
        ctx->impl.timing = enabled != 0;
        ctx->impl.count_tests = enabled >= 2;
    });
}

int hpd_context_set_graph(hpd_context* ctx, int enabled) {
    return guarded([&] {
        if (!ctx) throw Error(HPD_EINVAL, "context is NULL");
        Context& c = ctx->impl;
        c.graph = enabled != 0;
        if (!c.graph && c.graph_entry.exec) {
            hpd::DeviceGuard g(c.device);
            HPD_HIP(hipStreamSynchronize(c.stream));
            (void)hipGraphExecDestroy(c.graph_entry.exec);
            c.graph_entry = Context::GraphEntry{};
        }
    });
}

int hpd_context_get_graph_stats(const hpd_context* ctx, uint64_t* launches, uint64_t* captures,
                                uint64_t* fallbacks) {
    return guarded([&] {
        if (!ctx || !launches || !captures || !fallbacks) throw Error(HPD_EINVAL, "NULL argument");
        *launches = ctx->impl.graph_launches;
        *captures = ctx->impl.graph_captures;
        *fallbacks = ctx->impl.graph_fallbacks;
    });
}

int hpd_context_set_open_pair_limit(hpd_context* ctx, uint64_t limit) {
    return guarded([&] {
        if (!ctx) throw Error(HPD_EINVAL, "context is NULL");
        ctx->impl.open_pair_limit = limit;
    });
}

int hpd_context_set_work_split(hpd_context* ctx, int32_t sparse_max, int sparse_core) {
    return guarded([&] {
        if (!ctx) throw Error(HPD_EINVAL, "context is NULL");
        if (sparse_max < 0 || sparse_max > 64)
            throw Error(HPD_EINVAL, "sparse_max must be in [0, 64]");
        ctx->impl.sparse_max = sparse_max;
        ctx->impl.sparse_core = sparse_core != 0;
    });
}

int hpd_context_set_box_split(hpd_context* ctx, int32_t parts) {
    return guarded([&] {
        if (!ctx) throw Error(HPD_EINVAL, "context is NULL");
        if (parts < 0 || parts > 8) throw Error(HPD_EINVAL, "box split must be in [0, 8]");
        ctx->impl.box_split = parts;
    });
}

int hpd_context_get_box_split(const hpd_context* ctx, int32_t* parts) {
    return guarded([&] {
        if (!ctx || !parts) throw Error(HPD_EINVAL, "NULL argument");
        *parts = ctx->impl.box_split;
    });
}

int hpd_context_get_work_split(const hpd_context* ctx, int32_t* sparse_max, int* sparse_core) {
    return guarded([&] {
        if (!ctx || !sparse_max || !sparse_core) throw Error(HPD_EINVAL, "NULL argument");
        *sparse_max = ctx->impl.sparse_max;
        *sparse_core = ctx->impl.sparse_core ? 1 : 0;
    });
}

int hpd_context_get_stats(const hpd_context* ctx, hpd_run_stats* out) {
    return guarded([&] {
        if (!ctx || !out) throw Error(HPD_EINVAL, "NULL argument");
        *out = ctx->impl.stats;
    });
}

int hpd_cluster_device(hpd_context* ctx, int dtype, const void* data, int64_t n, int32_t d,
                       float eps, uint64_t min_pts, int64_t* labels_out, void* stream) {
    return guarded([&] {
        hpd::validate(ctx ? &ctx->impl : nullptr, dtype, data, n, d, eps, labels_out);
        Context& c = ctx->impl;
        c.stats = hpd_run_stats{};
        c.stats.n = n;
        c.stats.d = d;
        if (n == 0) return;
        hpd::DeviceGuard g(c.device);
        hipStream_t s = stream ? static_cast<hipStream_t>(stream) : c.stream;
        const int64_t offsets[2] = {0, n};
        hpd::run_any(c, dtype, data, n, d, offsets, 1, &eps, &min_pts, labels_out, s);
    });
}

int hpd_cluster_device_noalloc(hpd_context* ctx, int dtype, const void* data, int64_t n,
                               int32_t d, float eps, uint64_t min_pts, int64_t* labels_out,
                               void* stream) {
    return guarded([&] {
        hpd::validate(ctx ? &ctx->impl : nullptr, dtype, data, n, d, eps, labels_out);
        Context& c = ctx->impl;
        c.stats = hpd_run_stats{};
        c.stats.n = n;
        c.stats.d = d;
        if (n == 0) return;
        // the workspace of the main arena, checked before anything runs; the
        // neighbour tables and work lists take the rest and are checked when
        // their sizes are known (before any label is written)
        const size_t need = hpd::workspace_any(dtype, n, d, c.border_rule == HPD_BORDER_ONE_THREAD);
        if (need > hpd::kScratchBytes)
            throw Error(HPD_EUNSUPPORTED,
                        "hpd_cluster_device_noalloc: " + std::to_string(n) + " rows of " +
                            std::to_string(d) + " dimensions need " + std::to_string(need) +
                            " bytes of workspace; its static scratch holds " +
                            std::to_string(hpd::kScratchBytes) +
                            " bytes (use hpd_cluster_device for larger inputs)");
        hpd::DeviceGuard g(c.device);
        void* base = hpd::scratch_of(c.device);
        if (!base) throw Error(HPD_EDEVICE, "no scratch address for this device");
        hpd::FixedWorkspace ws(c, base, hpd::align_up(need, 256), hpd::kScratchBytes);
        hipStream_t s = stream ? static_cast<hipStream_t>(stream) : c.stream;
        const int64_t offsets[2] = {0, n};
        hpd::run_any(c, dtype, data, n, d, offsets, 1, &eps, &min_pts, labels_out, s);
    });
}

int hpd_cluster(hpd_context* ctx, int dtype, const void* data, int64_t n, int32_t d, float eps,
                uint64_t min_pts, int64_t* labels_out) {
    return guarded([&] {
        hpd::validate(ctx ? &ctx->impl : nullptr, dtype, data, n, d, eps, labels_out);
        Context& c = ctx->impl;
        c.stats = hpd_run_stats{};
        c.stats.n = n;
        c.stats.d = d;
        if (n == 0) return;
        hpd::DeviceGuard g(c.device);
        const size_t row_bytes = hpd::dtype_size(dtype) * static_cast<size_t>(d);
        const size_t in_bytes = row_bytes * static_cast<size_t>(n);
        const size_t out_bytes = sizeof(int64_t) * static_cast<size_t>(n);
        // input rows and output labels live in their own grow-only buffer
        c.io.reserve(hpd::align_up(in_bytes, 256) + out_bytes + 512);
        void* din = c.io.take(in_bytes);
        int64_t* dout = c.io.take_n<int64_t>(static_cast<size_t>(n));
        HPD_HIP(hipMemcpyAsync(din, data, in_bytes, hipMemcpyHostToDevice, c.stream));
        const int64_t offsets[2] = {0, n};
        hpd::run_any(c, dtype, din, n, d, offsets, 1, &eps, &min_pts, dout, c.stream);
        HPD_HIP(hipMemcpyAsync(labels_out, dout, out_bytes, hipMemcpyDeviceToHost, c.stream));
        HPD_HIP(hipStreamSynchronize(c.stream));
    });
}

static void validate_batch(const hpd_context* ctx, int dtype, const void* data,
                           const int64_t* offsets, int32_t njobs, int32_t d, const float* eps,
                           const uint64_t* min_pts, const void* labels) {
    if (!ctx) throw Error(HPD_EINVAL, "context is NULL");
    if (njobs < 0) throw Error(HPD_EINVAL, "the number of jobs must not be negative");
    if (njobs == 0) return;
    if (!offsets || !eps || !min_pts) throw Error(HPD_EINVAL, "offsets, eps and min_pts must not be NULL");
    if (offsets[0] != 0) throw Error(HPD_EINVAL, "offsets[0] must be 0");
    for (int32_t j = 0; j < njobs; ++j) {
        if (offsets[j + 1] < offsets[j]) throw Error(HPD_EINVAL, "offsets must not decrease");
        if (!(eps[j] > 0.0f))
            throw Error(HPD_EINVAL, "epsilon needs to be positive (job " + std::to_string(j) + ")");
    }
    hpd::validate(&ctx->impl, dtype, data, offsets[njobs], d, 1.0f, labels);
}

int hpd_cluster_batch_device(hpd_context* ctx, int dtype, const void* data,
                             const int64_t* offsets, int32_t njobs, int32_t d, const float* eps,
                             const uint64_t* min_pts, int64_t* labels_out, void* stream) {
    return guarded([&] {
        validate_batch(ctx, dtype, data, offsets, njobs, d, eps, min_pts, labels_out);
        Context& c = ctx->impl;
        c.stats = hpd_run_stats{};
        const int64_t n = njobs ? offsets[njobs] : 0;
        c.stats.n = n;
        c.stats.d = d;
        if (n == 0) return;
        hpd::DeviceGuard g(c.device);
        hipStream_t s = stream ? static_cast<hipStream_t>(stream) : c.stream;
        hpd::run_any(c, dtype, data, n, d, offsets, njobs, eps, min_pts, labels_out, s);
    });
}

int hpd_cluster_batch(hpd_context* ctx, int dtype, const void* data, const int64_t* offsets,
                      int32_t njobs, int32_t d, const float* eps, const uint64_t* min_pts,
                      int64_t* labels_out) {
    return guarded([&] {
        validate_batch(ctx, dtype, data, offsets, njobs, d, eps, min_pts, labels_out);
        Context& c = ctx->impl;
        c.stats = hpd_run_stats{};
        const int64_t n = njobs ? offsets[njobs] : 0;
        c.stats.n = n;
        c.stats.d = d;
        if (n == 0) return;
        hpd::DeviceGuard g(c.device);
        const size_t in_bytes = hpd::dtype_size(dtype) * static_cast<size_t>(d) * static_cast<size_t>(n);
        const size_t out_bytes = sizeof(int64_t) * static_cast<size_t>(n);
        c.io.reserve(hpd::align_up(in_bytes, 256) + out_bytes + 512);
        void* din = c.io.take(in_bytes);
        int64_t* dout = c.io.take_n<int64_t>(static_cast<size_t>(n));
        HPD_HIP(hipMemcpyAsync(din, data, in_bytes, hipMemcpyHostToDevice, c.stream));
        hpd::run_any(c, dtype, din, n, d, offsets, njobs, eps, min_pts, dout, c.stream);
        HPD_HIP(hipMemcpyAsync(labels_out, dout, out_bytes, hipMemcpyDeviceToHost, c.stream));
        HPD_HIP(hipStreamSynchronize(c.stream));
    });
}

int hpd_check_neighbor_rows(uint64_t neighbor_rows) {
    return guarded([&] { hpd::check_neighbor_rows(neighbor_rows); });
}

int hpd_device_alloc(hpd_context* ctx, size_t bytes, void** out) {
    return guarded([&] {
        if (!ctx || !out) throw Error(HPD_EINVAL, "NULL argument");
        *out = nullptr;
        hpd::DeviceGuard g(ctx->impl.device);
        HPD_HIP(hipMalloc(out, bytes > 0 ? bytes : 1));
    });
}

int hpd_device_free(hpd_context* ctx, void* ptr) {
    return guarded([&] {
        if (!ctx) throw Error(HPD_EINVAL, "context is NULL");
        if (!ptr) return;
        hpd::DeviceGuard g(ctx->impl.device);
        HPD_HIP(hipStreamSynchronize(ctx->impl.stream));
        HPD_HIP(hipFree(ptr));
    });
}

int hpd_memcpy_to_device(hpd_context* ctx, void* dst, const void* src, size_t bytes) {
    return guarded([&] {
        if (!ctx || (bytes && (!dst || !src))) throw Error(HPD_EINVAL, "NULL argument");
        hpd::DeviceGuard g(ctx->impl.device);
        HPD_HIP(hipMemcpyAsync(dst, src, bytes, hipMemcpyHostToDevice, ctx->impl.stream));
        HPD_HIP(hipStreamSynchronize(ctx->impl.stream));
    });
}

int hpd_memcpy_to_host(hpd_context* ctx, void* dst, const void* src, size_t bytes) {
    return guarded([&] {
        if (!ctx || (bytes && (!dst || !src))) throw Error(HPD_EINVAL, "NULL argument");
        hpd::DeviceGuard g(ctx->impl.device);
        HPD_HIP(hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToHost, ctx->impl.stream));
        HPD_HIP(hipStreamSynchronize(ctx->impl.stream));
    });
}

int hpd_context_stream(hpd_context* ctx, void** stream_out) {
    return guarded([&] {
        if (!ctx || !stream_out) throw Error(HPD_EINVAL, "NULL argument");
        *stream_out = static_cast<void*>(ctx->impl.stream);
    });
}

int hpd_context_synchronize(hpd_context* ctx) {
    return guarded([&] {
        if (!ctx) throw Error(HPD_EINVAL, "context is NULL");
        hpd::DeviceGuard g(ctx->impl.device);
        HPD_HIP(hipStreamSynchronize(ctx->impl.stream));
    });
}

}  // extern "C"
