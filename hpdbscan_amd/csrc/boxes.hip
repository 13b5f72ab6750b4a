// Sub-boxes of the eps-grid cells and the box-level union of core points.
//
// Every occupied cell is split into k^D sub-boxes along the same scaled
// coordinate the cell index uses, v = (x - min) * (1/eps):
//   sub_d = clamp(floor(v_d * k) - k * floor(v_d), 0, k - 1)
// with k = 2 for D <= 3 and k = 3 for D <= 8, so a box is at most eps/k wide
// and its diagonal at most 0.94 eps.  Rows are regrouped by (cell, box)
// inside each cell; the reference's sorted position of every row is kept
// beside it (the cluster ids are smallest positions, not slots).
//
// A box is "tight" when the reference's own squared-distance expression
// evaluated on the box extents, dist2(max - min), is <= EPS2.  Every
// rounding step of that expression (subtract, square, the summation tree,
// the flush of tiny values) is monotone in its inputs and |p_d - q_d| <=
// max_d - min_d for any two members, so every pair of members of a tight
// box passes the reference's within-eps test, and they share a cell, so they
// are each other's candidates.  Hence:
//   * a tight box with >= minPts rows makes all its rows core;
//   * all cores of a tight box lie in one cluster.
// The union of the cores is therefore computed on boxes: two boxes with
// cores are joined when some core pair across them is within eps (tested
// with the reference's expression, stopping at the first hit), unless they
// are already joined; a core row farther than eps from the other box's
// bounding box takes no part in the test.  Box pairs whose bounding boxes are
// farther apart than eps by the same monotone expression (box_gap) cannot hold
// such a pair and are skipped.
#include <algorithm>
#include <climits>

#include "boxes.hpp"
#include "hpdbscan_capi.h"
#include "collect.hpp"
#include "common.hpp"
#include "grid.hpp"
#include "index.hpp"
#include "internal.hpp"
#include "visit.hpp"

namespace hpd {

namespace {

constexpr int kThreads = 256;
constexpr int kWavesPerBlock = kThreads / kWave;
inline unsigned blocks_for(int64_t n, int t) { return static_cast<unsigned>((n + t - 1) / t); }

// Rows in slot order: coordinates (SoA); with it the bounding box of every
// box (ordered keys).  A block of kThreads slots reduces its boxes in LDS
// (box ids are consecutive in slot order, so a box's LDS entry is its id less
// the block's first box): a box inside the block is stored by the block; the
// block's first box when it started in an earlier block, and its last box
// when it goes on past the block, leave the block's share in
// part[(2 * block + 0 / 1) * 2D ..] for k_box_span.  No global atomics: a
// box of a million rows would otherwise take thousands of them on one
// address.  With pts null the coordinates are already in soa (the sort
// moved them) and only the bounding boxes are made.
template <typename T, int D>
__global__ __launch_bounds__(kThreads) void k_gather_boxes(
    const T* __restrict__ pts, int64_t n, const uint32_t* __restrict__ inrow_of_slot,
    T* __restrict__ soa, int64_t ld, const int32_t* __restrict__ box_of_slot,
    const int32_t* __restrict__ bstart, Span<T>* __restrict__ bbox, OrdKey<T>* __restrict__ part) {
    using U = OrdKey<T>;
    __shared__ U slo[kThreads][D];
    __shared__ U shi[kThreads][D];
    const int64_t blk0 = static_cast<int64_t>(blockIdx.x) * kThreads;
    const int64_t s = blk0 + threadIdx.x;
    const bool valid = s < n;
#pragma unroll
    for (int j = 0; j < D; ++j) {
        slo[threadIdx.x][j] = static_cast<U>(~U(0));
        shi[threadIdx.x][j] = U(0);
    }
    const int32_t b_first = box_of_slot[blk0];  // the block's first box
    int32_t b = -1 - lane_id();  // distinct keys for lanes past the end
    T x[D];
    if (valid && !pts) {
        b = box_of_slot[s];
#pragma unroll
        for (int j = 0; j < D; ++j) x[j] = soa[static_cast<int64_t>(j) * ld + s];
    } else if (valid) {
        const uint32_t row = inrow_of_slot[s];
        b = box_of_slot[s];
#pragma unroll
        for (int j = 0; j < D; ++j) {
            x[j] = pts[static_cast<int64_t>(row) * D + j];
            soa[static_cast<int64_t>(j) * ld + s] = x[j];
        }
    } else {
#pragma unroll
        for (int j = 0; j < D; ++j) x[j] = T(0);
    }
    __syncthreads();
    // every lane takes part in the shuffles; the head lane of each run in the
    // wave (lane 0 included) adds the run's extremes to the box's LDS entry
    const bool head = valid && run_head(b);
#pragma unroll
    for (int j = 0; j < D; ++j) {
        const U k = ord_key(x[j]);
        const U lo = run_suffix_min<U>(k, b);
        const U hi = run_suffix_max<U>(k, b);
        if (head) {
            atomicMin(&slo[b - b_first][j], lo);
            atomicMax(&shi[b - b_first][j], hi);
        }
    }
    __syncthreads();
    const int64_t blk1 = blk0 + kThreads < n ? blk0 + kThreads : n;  // end of the block's slots
    const int32_t nruns = box_of_slot[blk1 - 1] - b_first + 1;
    for (int t = threadIdx.x; t < nruns; t += kThreads) {
        const int32_t bb = b_first + t;
        const bool starts = bstart[bb] >= blk0;
        const bool ends = bstart[bb + 1] <= blk1;
        if (starts && ends) {
#pragma unroll
            for (int j = 0; j < D; ++j)
                bbox[static_cast<int64_t>(bb) * D + j] = {ord_val(slo[t][j]), ord_val(shi[t][j])};
            continue;
        }
        U* dst = &part[(2 * static_cast<int64_t>(blockIdx.x) + (starts ? 1 : 0)) * D * 2];
#pragma unroll
        for (int j = 0; j < D; ++j) {
            dst[2 * j] = slo[t][j];
            dst[2 * j + 1] = shi[t][j];
        }
    }
}

// Bounding boxes only, the coordinates being in slot order already (the
// sort carried them): k_gather_boxes' reduction over tiles of kBoundsRows
// wave-segments per thread (a tile of kThreads * kBoundsRows slots per
// block, all of a thread's slots loaded first), so that the LDS set-up,
// the barriers and the stores of a block are shared by four times the
// slots.  Rows of at most 8 bytes (LDS: 2 * tile * D ordered keys).
constexpr int kBoundsRows = 4;
constexpr int kBoundsTile = kThreads * kBoundsRows;

template <typename T, int D>
__global__ __launch_bounds__(kThreads) void k_box_bounds(
    const T* __restrict__ soa, int64_t ld, int64_t n, const int32_t* __restrict__ box_of_slot,
    const int32_t* __restrict__ bstart, Span<T>* __restrict__ bbox, OrdKey<T>* __restrict__ part) {
    using U = OrdKey<T>;
    static_assert(D * sizeof(T) <= 8, "rows of at most 8 bytes");
    __shared__ U slo[kBoundsTile][D];
    __shared__ U shi[kBoundsTile][D];
    const int64_t blk0 = static_cast<int64_t>(blockIdx.x) * kBoundsTile;
    for (int e = threadIdx.x; e < kBoundsTile; e += kThreads) {
#pragma unroll
        for (int j = 0; j < D; ++j) {
            slo[e][j] = static_cast<U>(~U(0));
            shi[e][j] = U(0);
        }
    }
    const int32_t b_first = box_of_slot[blk0];  // the block's first box
    const int w = static_cast<int>(threadIdx.x >> 6);
    // segment k of wave w: slots blk0 + (k * kWavesPerBlock + w) * 64 + lane
    int32_t b[kBoundsRows];
    T x[kBoundsRows][D];
#pragma unroll
    for (int k = 0; k < kBoundsRows; ++k) {
        const int64_t s = blk0 + (static_cast<int64_t>(k) * kWavesPerBlock + w) * kWave + lane_id();
        const bool valid = s < n;
        b[k] = valid ? box_of_slot[s] : -1 - static_cast<int32_t>(lane_id());
#pragma unroll
        for (int j = 0; j < D; ++j) x[k][j] = valid ? soa[static_cast<int64_t>(j) * ld + s] : T(0);
    }
    const int64_t blk1 = blk0 + kBoundsTile < n ? blk0 + kBoundsTile : n;
    __syncthreads();
    if (b_first == box_of_slot[blk1 - 1]) {
        // the whole tile is one box (large boxes): each thread's slots,
        // then one reduction per wave, then one LDS merge per wave
        U lo[D], hi[D];
#pragma unroll
        for (int j = 0; j < D; ++j) {
            lo[j] = static_cast<U>(~U(0));
            hi[j] = U(0);
        }
#pragma unroll
        for (int k = 0; k < kBoundsRows; ++k) {
            if (b[k] < 0) continue;
#pragma unroll
            for (int j = 0; j < D; ++j) {
                const U key = ord_key(x[k][j]);
                lo[j] = key < lo[j] ? key : lo[j];
                hi[j] = key > hi[j] ? key : hi[j];
            }
        }
#pragma unroll
        for (int j = 0; j < D; ++j) {
#pragma unroll
            for (int o = 32; o > 0; o >>= 1) {
                const U a = static_cast<U>(__shfl_xor(lo[j], o, 64));
                const U z = static_cast<U>(__shfl_xor(hi[j], o, 64));
                lo[j] = a < lo[j] ? a : lo[j];
                hi[j] = z > hi[j] ? z : hi[j];
            }
            if (lane_id() == 0) {
                atomicMin(&slo[0][j], lo[j]);
                atomicMax(&shi[0][j], hi[j]);
            }
        }
    } else {
#pragma unroll
        for (int k = 0; k < kBoundsRows; ++k) {
            // the head lane of each run of the segment adds the run's extremes
            const bool head = b[k] >= 0 && run_head(b[k]);
#pragma unroll
            for (int j = 0; j < D; ++j) {
                const U key = ord_key(x[k][j]);
                const U lo = run_suffix_min<U>(key, b[k]);
                const U hi = run_suffix_max<U>(key, b[k]);
                if (head) {
                    atomicMin(&slo[b[k] - b_first][j], lo);
                    atomicMax(&shi[b[k] - b_first][j], hi);
                }
            }
        }
    }
    __syncthreads();
    const int32_t nruns = box_of_slot[blk1 - 1] - b_first + 1;
    for (int t = threadIdx.x; t < nruns; t += kThreads) {
        const int32_t bb = b_first + t;
        const bool starts = bstart[bb] >= blk0;
        const bool ends = bstart[bb + 1] <= blk1;
        if (starts && ends) {
#pragma unroll
            for (int j = 0; j < D; ++j)
                bbox[static_cast<int64_t>(bb) * D + j] = {ord_val(slo[t][j]), ord_val(shi[t][j])};
            continue;
        }
        U* dst = &part[(2 * static_cast<int64_t>(blockIdx.x) + (starts ? 1 : 0)) * D * 2];
#pragma unroll
        for (int j = 0; j < D; ++j) {
            dst[2 * j] = slo[t][j];
            dst[2 * j + 1] = shi[t][j];
        }
    }
}

// Bounding boxes of the boxes that span blocks of k_gather_boxes: one wave
// per block; the wave of the block where such a box starts combines the
// block's share (its last run) with the shares of the following blocks (their
// first runs) up to the box's last block.
template <typename T, int D>
__global__ __launch_bounds__(kThreads) void k_box_span(int64_t n, int64_t nblocks, int64_t tile,
                                                       const int32_t* __restrict__ box_of_slot,
                                                       const int32_t* __restrict__ bstart,
                                                       const OrdKey<T>* __restrict__ part,
                                                       Span<T>* __restrict__ bbox) {
    using U = OrdKey<T>;
    const int64_t blk = static_cast<int64_t>(blockIdx.x) * kWavesPerBlock + (threadIdx.x >> 6);
    if (blk >= nblocks) return;
    const int64_t blk0 = blk * tile;
    const int64_t blk1 = blk0 + tile < n ? blk0 + tile : n;
    const int32_t b = box_of_slot[blk1 - 1];
    const int64_t b0 = bstart[b], b1 = bstart[b + 1];
    if (b0 < blk0 || b1 <= blk1) return;  // not a box that starts here and goes on
    const int64_t last = (b1 - 1) / tile;
    U lo[D], hi[D];
#pragma unroll
    for (int j = 0; j < D; ++j) {
        lo[j] = static_cast<U>(~U(0));
        hi[j] = U(0);
    }
    for (int64_t k = blk + lane_id(); k <= last; k += kWave) {
        const U* src = &part[(2 * k + (k == blk ? 1 : 0)) * D * 2];
#pragma unroll
        for (int j = 0; j < D; ++j) {
            lo[j] = min(lo[j], src[2 * j]);
            hi[j] = max(hi[j], src[2 * j + 1]);
        }
    }
#pragma unroll
    for (int j = 0; j < D; ++j) {
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) {
            lo[j] = min(lo[j], static_cast<U>(__shfl_xor(lo[j], o, 64)));
            hi[j] = max(hi[j], static_cast<U>(__shfl_xor(hi[j], o, 64)));
        }
    }
    if (lane_id() == 0) {
#pragma unroll
        for (int j = 0; j < D; ++j)
            bbox[static_cast<int64_t>(b) * D + j] = {ord_val(lo[j]), ord_val(hi[j])};
    }
}

// Boxes and occupied cells from the sorted keys, in two passes over them: the
// box and cell starts of every block's run of tiles are counted, then each
// block adds up the counts of the blocks before it and numbers its own starts.
// Bound by reading the keys twice and writing the box of every slot.  (Flag
// arrays over the slots and over the boxes, each scanned in two launches, were
// six launches more.  Whole calls, before and now: 100k rows 398 -> 362 us, 100M
// 6.18 -> 5.53 ms, 4096 clouds of 8k rows 37.4 -> 36.0 ms.)
constexpr int kTablePer = 8;  // keys per lane and tile, in wave segments of 64
constexpr int kTableTile = kThreads * kTablePer;
// blocks at most: each reads the counts of all before it (8 bytes a block)
constexpr int64_t kTableBlocks = 2048;
inline int64_t table_tiles(int64_t n) { return (n + kTableTile - 1) / kTableTile; }
inline int table_run(int64_t n) {
    return static_cast<int>((table_tiles(n) + kTableBlocks - 1) / kTableBlocks);
}

// The keys of a wave's part of the tile at t (segment k of it: 64 keys from
// first + k * 64), and per segment the lanes whose key starts a box, a cell.
template <typename K>
struct TableTile {
    K key[kTablePer];
    uint64_t box[kTablePer], cell[kTablePer];
    int64_t first;
    __device__ __forceinline__ TableTile(const K* __restrict__ keys, int64_t n, int64_t t,
                                         int shift) {
        first = t + static_cast<int64_t>(threadIdx.x >> 6) * (kWave * kTablePer);
        K before[kTablePer];
#pragma unroll
        for (int k = 0; k < kTablePer; ++k) {
            const int64_t i = first + k * kWave + lane_id();
            key[k] = i < n ? keys[i] : K(0);
            before[k] = i < n && i > 0 ? keys[i - 1] : K(0);
        }
#pragma unroll
        for (int k = 0; k < kTablePer; ++k) {
            const int64_t i = first + k * kWave + lane_id();
            box[k] = ballot(i < n && (i == 0 || key[k] != before[k]));
            cell[k] = ballot(i < n && (i == 0 || (key[k] >> shift) != (before[k] >> shift)));
        }
    }
    // box starts, cell starts of the wave's part
    __device__ __forceinline__ uint2 count() const {
        uint2 c = make_uint2(0, 0);
#pragma unroll
        for (int k = 0; k < kTablePer; ++k) {
            c.x += static_cast<uint32_t>(__popcll(box[k]));
            c.y += static_cast<uint32_t>(__popcll(cell[k]));
        }
        return c;
    }
};

template <typename K>
__global__ __launch_bounds__(kThreads) void k_table_count(const K* __restrict__ keys, int64_t n,
                                                          int shift, int run,
                                                          uint2* __restrict__ sums) {
    __shared__ uint2 part[kWavesPerBlock];
    uint2 c = make_uint2(0, 0);
    const int64_t t0 = static_cast<int64_t>(blockIdx.x) * run * kTableTile;
    for (int r = 0; r < run && t0 + r * kTableTile < n; ++r) {
        const TableTile<K> tile(keys, n, t0 + r * kTableTile, shift);
        const uint2 k = tile.count();
        c.x += k.x;
        c.y += k.y;
    }
    if (lane_id() == 0) part[threadIdx.x >> 6] = c;
    __syncthreads();
    if (threadIdx.x == 0) {
        c = make_uint2(0, 0);
#pragma unroll
        for (int w = 0; w < kWavesPerBlock; ++w) {
            c.x += part[w].x;
            c.y += part[w].y;
        }
        sums[blockIdx.x] = c;
    }
}

template <typename K>
__global__ __launch_bounds__(kThreads) void k_table_write(
    const K* __restrict__ keys, int64_t n, int shift, int run, const uint2* __restrict__ sums,
    int32_t* __restrict__ box_of_slot, int32_t* __restrict__ bstart, int32_t* __restrict__ bcell,
    K* __restrict__ ucell, int32_t* __restrict__ ustart, int32_t* __restrict__ cbox,
    int32_t* __restrict__ ctab, uint32_t* __restrict__ nbox_dev,
    uint32_t* __restrict__ ncells_dev) {
    __shared__ uint2 part[kWavesPerBlock];
    const int w = static_cast<int>(threadIdx.x >> 6);
    // sum over the waves; own: the waves before this one
    auto wave_sums = [&](uint2 c, uint2& own) {
        __syncthreads();
        if (lane_id() == 0) part[w] = c;
        __syncthreads();
        uint2 all = make_uint2(0, 0);
        own = make_uint2(0, 0);
#pragma unroll
        for (int k = 0; k < kWavesPerBlock; ++k) {
            if (k < w) {
                own.x += part[k].x;
                own.y += part[k].y;
            }
            all.x += part[k].x;
            all.y += part[k].y;
        }
        return all;
    };
    uint2 at = make_uint2(0, 0), own;
    for (unsigned int j = threadIdx.x; j < blockIdx.x; j += kThreads) {
        at.x += sums[j].x;
        at.y += sums[j].y;
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
        at.x += __shfl_xor(at.x, o, 64);
        at.y += __shfl_xor(at.y, o, 64);
    }
    at = wave_sums(at, own);
    const uint64_t le = lanemask_lt() | (uint64_t{1} << lane_id());
    const int64_t t0 = static_cast<int64_t>(blockIdx.x) * run * kTableTile;
    for (int r = 0; r < run && t0 + r * kTableTile < n; ++r) {
        const TableTile<K> tile(keys, n, t0 + r * kTableTile, shift);
        const uint2 all = wave_sums(tile.count(), own);
        uint32_t b0 = at.x + own.x, u0 = at.y + own.y;
#pragma unroll
        for (int k = 0; k < kTablePer; ++k) {
            const int64_t i = tile.first + k * kWave + lane_id();
            const int32_t b = static_cast<int32_t>(
                b0 + static_cast<uint32_t>(__popcll(tile.box[k] & le)) - 1u);
            if (i < n) box_of_slot[i] = b;
            if ((tile.box[k] >> lane_id()) & 1) {
                const int32_t u = static_cast<int32_t>(
                    u0 + static_cast<uint32_t>(__popcll(tile.cell[k] & le)) - 1u);
                bstart[b] = static_cast<int32_t>(i);
                bcell[b] = u;
                if ((tile.cell[k] >> lane_id()) & 1) {
                    const K id = tile.key[k] >> shift;
                    ucell[u] = id;
                    ustart[u] = static_cast<int32_t>(i);
                    cbox[u] = b;
                    if (ctab) ctab[static_cast<uint64_t>(id)] = u;
                }
            }
            b0 += static_cast<uint32_t>(__popcll(tile.box[k]));
            u0 += static_cast<uint32_t>(__popcll(tile.cell[k]));
        }
        at.x += all.x;
        at.y += all.y;
    }
    if (blockIdx.x == gridDim.x - 1 && threadIdx.x == 0) {
        bstart[at.x] = static_cast<int32_t>(n);
        ustart[at.y] = static_cast<int32_t>(n);
        cbox[at.y] = static_cast<int32_t>(at.x);
        *nbox_dev = at.x;
        *ncells_dev = at.y;
    }
}

// rows of a box from which its pairs of the union go by parts (k_box_union)
constexpr int kHeavyRows = 2048;

// flags per box: tight (dist2(extent) <= EPS2 in the reference's order),
// full, in a cell that can hold cores
template <typename T, int D>
__global__ __launch_bounds__(kThreads) void k_box_tight(const Span<T>* __restrict__ bbox,
                                                        Count nbox_c,
                                                        const int32_t* __restrict__ bstart,
                                                        const int32_t* __restrict__ bcell,
                                                        const int32_t* __restrict__ job_of_cell,
                                                        const JobParams<T>* __restrict__ jobs,
                                                        const uint8_t* __restrict__ cell_core,
                                                        uint8_t* __restrict__ btight,
                                                        unsigned int* __restrict__ nloose,
                                                        int32_t large,
                                                        unsigned int* __restrict__ nlarge) {
    const int32_t nbox = static_cast<int32_t>(nbox_c.get());
    const int32_t b = static_cast<int32_t>(blockIdx.x) * kThreads + threadIdx.x;
    if (b >= nbox) return;
    const int32_t u = bcell[b];
    const JobParams<T>& jp = jobs[job_of_cell[u]];
    T lo[D], hi[D];
#pragma unroll
    for (int j = 0; j < D; ++j) {
        lo[j] = bbox[static_cast<int64_t>(b) * D + j].lo;
        hi[j] = bbox[static_cast<int64_t>(b) * D + j].hi;
    }
    const bool tight = within<D>(hi, lo, jp.eps2);
    const int32_t size = bstart[b + 1] - bstart[b];
    // bit 0: tight; bit 1: tight and at least minPts rows (all rows core)
    btight[b] = static_cast<uint8_t>((tight ? 1 : 0) |
                                     ((tight && static_cast<uint32_t>(size) >= jp.min_pts) ? 2 : 0) |
                                     (cell_core[u] ? 4 : 0));
    if (!tight && size > 1) atomicAdd(nloose, 1u);
    if (size > large) atomicAdd(&nlarge[0], 1u);
    if (size > kHeavyRows) atomicAdd(&nlarge[1], 1u);
}

// Whether a core row of a box, [q0, q1), is within eps of the row of a lane
// in `act` (wave-uniform answer, first hit stops).
template <typename T, int D>
__device__ __forceinline__ bool any_pair(const T* __restrict__ soa, int64_t ld,
                                         const uint8_t* __restrict__ core, int32_t q0, int32_t q1,
                                         const T* pc, bool act, T eps2) {
    const uint64_t rows = ballot(act);
    if (walk_wide(rows, q1 - q0))
        return __any(wide_any<T, D>(soa, ld, core, q0, q1, pc, eps2, rows, true));
    bool hit = false;
    auto body = [&](int32_t, const T* qc, uint8_t cq, int32_t) {
        if (cq && act && within<D>(pc, qc, eps2)) hit = true;
    };
    auto stop = [&] { return static_cast<bool>(__any(hit)); };
    return visit_range<T, D>(soa, ld, core, nullptr, q0, q1, body, stop);
}

// Whether a core row of slots [s0, s1) is within eps of a core row of box b2
// (slots [q0, q1)), by the whole wave (every argument wave-uniform): 64 rows
// of [s0, s1) at a time on the lanes; a row within eps of the whole box
// answers at once, one farther than eps from its bounding box is left out,
// the others meet the box's rows.
template <typename T, int D>
__device__ __forceinline__ bool wave_pair(const T* __restrict__ soa, int64_t ld,
                                          const uint8_t* __restrict__ core,
                                          const Span<T>* __restrict__ bbox, int32_t s0, int32_t s1,
                                          int32_t b2, int32_t q0, int32_t q1, T eps2) {
    for (int32_t c = s0; c < s1; c += kWave) {
        const int32_t p = c + lane_id();
        const bool pcore = p < s1 && core[p];
        if (!__any(pcore)) continue;
        T pc[D];
        load_row<T, D>(soa, ld, pcore ? p : c, pc);
        T gmin2, gmax2;
        point_box<T, D>(bbox, b2, pc, gmin2, gmax2);
        const bool act = pcore && gmin2 <= eps2;
        if (__any(act && gmax2 <= eps2)) return true;
        if (__any(act) && any_pair<T, D>(soa, ld, core, q0, q1, pc, act, eps2)) return true;
    }
    return false;
}

// The same by one lane, for boxes of few rows.
template <typename T, int D>
__device__ __forceinline__ bool lane_pair(const T* __restrict__ soa, int64_t ld,
                                          const uint8_t* __restrict__ core, int32_t s0, int32_t s1,
                                          int32_t q0, int32_t q1, T eps2) {
    for (int32_t p = s0; p < s1; ++p) {
        const bool cp = core[p] != 0;
        T pc[D];
        load_row<T, D>(soa, ld, p, pc);
        // (four rows side by side: their loads don't wait for each other)
        for (int32_t q = q0; q < q1; q += 4) {
            T qc[4][D];
            bool cq[4];
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                const int32_t at = min(q + k, q1 - 1);
                cq[k] = core[at] != 0;
                load_row<T, D>(soa, ld, at, qc[k]);
            }
            bool hit = false;
#pragma unroll
            for (int k = 0; k < 4; ++k) hit = hit || (cq[k] && within<D>(pc, qc[k], eps2));
            if (hit && cp) return true;
        }
    }
    return false;
}

// Whether one of the first and last rows of both boxes make such a pair.
template <typename T, int D>
__device__ __forceinline__ bool ends_pair(const T* __restrict__ soa, int64_t ld,
                                          const uint8_t* __restrict__ core, int32_t s0, int32_t s1,
                                          int32_t q0, int32_t q1, T eps2) {
    const int32_t p[2] = {s0, s1 - 1}, q[2] = {q0, q1 - 1};
    T pc[2][D], qc[2][D];
    uint8_t cp[2], cq[2];
#pragma unroll
    for (int k = 0; k < 2; ++k) {
        load_row<T, D>(soa, ld, p[k], pc[k]);
        load_row<T, D>(soa, ld, q[k], qc[k]);
        cp[k] = core[p[k]];
        cq[k] = core[q[k]];
    }
    bool hit = false;
#pragma unroll
    for (int k = 0; k < 4; ++k)
        hit = hit || (cp[k & 1] && cq[k >> 1] && within<D>(pc[k & 1], qc[k >> 1], eps2));
    return hit;
}

// The pair kernels below take the boxes with cores from blist, a group of G
// lanes per box, a neighbour box per lane (group_boxes); box pairs of up to
// kLanePair rows by rows are tested by their lane, larger ones by the wave.
// (4096 clouds, hook and join ms: 16 4.79, 32 4.83, 64 4.91, 256 11.4 before
// the first and last rows were tried first, 1024 13.2.)
constexpr int kLanePair = 16;
// Lanes per box: neighbourhoods grow with 3^D, and a group hands its lanes one
// box each per round of dependent loads.  Hook and join / union ms by lanes:
// 10M rows of 3 (8 lanes) 0.169 / 0.133, (16) 0.196 / 0.152, (32) 0.265 / 0.196;
// 5M of 4 (16) 0.299 / 0.614, (32) 0.243 / 0.624, (64) 0.286 / 0.673; 30k of 6
// doubles (16) 0.220 / 0.119, (32) 0.147 / 0.109, (64) 0.123 / 0.112.
template <int D>
constexpr int kPairGroup = D <= 3 ? 8 : D == 4 ? 32 : 64;
constexpr int kLinkRows = 4096;

// The same bounds (point_box) for the rows of two boxes: gap2 <= dist2(p, q)
// <= far2 for every pair of members.
template <typename T, int D>
__device__ __forceinline__ void box_gap(const Span<T>* __restrict__ bbox, int32_t b2,
                                        const Span<T>* mine, T& gap2, T& far2) {
    T g[D], f[D];
#pragma unroll
    for (int j = 0; j < D; ++j) {
        const Span<T> s = bbox[static_cast<int64_t>(b2) * D + j];
        g[j] = max(T(0), max(s.lo - mine[j].hi, mine[j].lo - s.hi));
        f[j] = max(s.hi - mine[j].lo, mine[j].hi - s.lo);
    }
    gap2 = sum2<D>(g);
    far2 = sum2<D>(f);
}

// Hook forest (kJoin false): every listed box points at some earlier box
// holding a core within eps of one of its cores, the own neighbour row
// searched first from the own cell on (any such box will do, and a box
// without one stays a root; boxes search from their first 64 rows and through
// the other box's first kLinkRows only, here and in the root join: a missed
// link is found by the exact union later).  bparent stays <=
// the box index, so the hooks form a forest whose trees are connected sets
// of boxes.
// Root join (kJoin): every root of that forest (blist) looks through its
// whole neighbourhood for the first box of another tree (rsnap) holding a
// within-eps core pair and joins the two trees (union-find, smaller root on
// top).  One round merges most trees of a cluster, so far fewer pairs stay
// open for the union.
// tag: bmincore (INT_MAX: no cores) for the hook, rsnap (-1) for the join.
template <typename T, int D, bool kJoin>
__global__ __launch_bounds__(kThreads) void k_box_link(const BoxArgs<T> a,
                                                       const uint32_t* __restrict__ roff,
                                                       const int2* __restrict__ rboxes,
                                                       const int32_t* __restrict__ tag,
                                                       const uint8_t* __restrict__ core,
                                                       const int32_t* __restrict__ blist,
                                                       const unsigned int* __restrict__ nlist_dev,
                                                       int32_t* bparent) {
    constexpr int G = kPairGroup<D>;
    constexpr int kPer = 64 / G;
    const int32_t nlist = uniform(static_cast<int32_t>(*nlist_dev));
    const int gl = lane_id() & (G - 1);
    const int grp = lane_id() / G;
    const Span<T>* bbox = static_cast<const Span<T>*>(a.bbox);
    for (int32_t base = first_wave() * kPer; base < nlist; base += wave_stride() * kPer) {
        const bool on = base + grp < nlist;
        const int32_t b = blist[on ? base + grp : nlist - 1];
        const int32_t s0 = a.bstart[b], s1 = a.bstart[b + 1];
        const int32_t u = a.bcell[b];
        const JobParams<T>& jp = a.jobs[a.njobs == 1 ? 0 : a.job_of_cell[u]];
        const T eps2 = jp.eps2;
        Span<T> mine[D];
#pragma unroll
        for (int j = 0; j < D; ++j) mine[j] = bbox[static_cast<int64_t>(b) * D + j];
        int32_t link = -1;  // equal over the group
        group_boxes<G>(on, static_cast<int32_t>(roff[u]), static_cast<int32_t>(roff[u + 1]),
                       a.rcenter[u], a.cbox[u], rboxes, 0, kJoin ? INT_MAX : b,
                       [&](bool valid, int32_t b2) {
            bool open = false, hit = false;
            int32_t q0 = 0, q1 = 0;
            if (valid) {
                const int32_t t = tag[b2];
                if (kJoin ? (t >= 0 && t != b) : t != INT_MAX) {
                    T gap2, far2;
                    box_gap<T, D>(bbox, b2, mine, gap2, far2);
                    open = gap2 <= eps2;
                    hit = far2 <= eps2;
                    q0 = a.bstart[b2];
                    q1 = a.bstart[b2 + 1];
                }
            }
            const uint64_t gmask = ((G < 64 ? (uint64_t{1} << G) : 0) - 1) << (grp * G);
            uint64_t hits = ballot(hit) & gmask;
            if (hits == 0 && open) {
                // the first and last rows of both boxes first: neighbouring
                // boxes mostly hold a pair among them, and a lane that runs
                // into a box without one holds up its wave
                hit = ends_pair<T, D>(a.soa, a.ld, core, s0, s1, q0, q1, eps2);
            }
            hits = ballot(hit) & gmask;
            if (hits == 0 && open) {
                const int64_t tests = static_cast<int64_t>(s1 - s0) * (q1 - q0);
                if (tests <= kLanePair) {
                    hit = lane_pair<T, D>(a.soa, a.ld, core, s0, s1, q0, q1, eps2);
                    open = false;
                }
            }
            const bool none = hits == 0;
            hits = none ? ballot(hit) & gmask : hits;
            // (the ballot is taken where `none` holds, which is equal over a
            // group: a group takes it whole and reads its own lanes only)
            bool done = hits != 0;
            for (uint64_t todo = ballot(open && !done); todo != 0; todo &= todo - 1) {
                const int j = static_cast<int>(__builtin_ctzll(todo));
                if ((ballot(done) >> j) & 1) continue;
                const int32_t t0 = bcast(s0, j);
                const int32_t v0 = bcast(q0, j);
                if (wave_pair<T, D>(a.soa, a.ld, core, bbox, t0, min(bcast(s1, j), t0 + kWave),
                                    bcast(b2, j), v0, min(bcast(q1, j), v0 + kLinkRows),
                                    bcast(eps2, j))) {
                    if (grp == j / G) {
                        done = true;
                        hits = uint64_t{1} << j;
                    }
                }
            }
            if (hits != 0) link = __shfl(b2, static_cast<int>(__builtin_ctzll(hits)), 64);
            return done;
        });
        if (on && gl == 0 && link >= 0) {
            if (kJoin) uf_unite(bparent, b, link);
            else bparent[b] = link;
        }
    }
}

// The boxes with cores of the cells whose own boxes and later neighbour boxes
// lie in different snapshot trees (rsnap) go to `list`: only they can have open
// pairs.  A group of lanes per cell, which ends at the first box of another
// tree; a cell's boxes share the neighbourhood, and most cells lie inside one
// tree.  From 4-D on and for many boxes: the neighbourhoods are large, or a launch
// is cheap beside them (union with this kernel and without, us: 5M rows of 4
// floats 203, 630; 30k of 6 doubles 33, 112; 4096 clouds of 3 3218, 4720; 10M
// rows of 3, 1.0M boxes, 116, 137; 100k of 3 60, 42; 300k of 2 38, 26).  Near the
// line it is the data that decides: blobs with 10 % noise of 3 by boxes 128k
// 75, 64; 224k 95, 83; 376k 123, 112; 942k 262, 250; of 2 174k 71, 61; 694k 124,
// 111; 1.3M 144, 147.  So between the line and about a million boxes such a
// cloud loses some 12 us (1 to 2 % of its call); the 10M rows gain a seventh of
// the union, the batch of clouds a third.
constexpr int64_t kMixedBoxes = 250000;
constexpr int kMixedStage = 512;  // list entries staged per wave
template <int D>
__global__ __launch_bounds__(kThreads) void k_mixed_cells(
    Count m_c, const int32_t* __restrict__ cbox, const uint32_t* __restrict__ roff,
    const int2* __restrict__ rboxes, const int32_t* __restrict__ rsnap, int32_t* __restrict__ list,
    unsigned int* __restrict__ count) {
    constexpr int G = kPairGroup<D>;
    constexpr int kPer = 64 / G;
    __shared__ int32_t stage[kWavesPerBlock][kMixedStage];
    __shared__ unsigned int left[kWavesPerBlock], at0;
    const int32_t m = uniform(static_cast<int32_t>(m_c.get()));
    const int w = static_cast<int>(threadIdx.x >> 6);
    const int gl = lane_id() & (G - 1);
    const int grp = lane_id() / G;
    const uint64_t gmask = ((G < 64 ? (uint64_t{1} << G) : 0) - 1) << (grp * G);
    unsigned int fill = 0;  // of the wave's stage
    for (int32_t base = first_wave() * kPer; base < m; base += wave_stride() * kPer) {
        const bool on = base + grp < m;
        const int32_t u = on ? base + grp : m - 1;
        const int32_t c0 = cbox[u], c1 = cbox[u + 1];
        const int32_t r0 = static_cast<int32_t>(roff[u]), r1 = static_cast<int32_t>(roff[u + 1]);
        int32_t lo = INT_MAX, hi = -1;
        for (int32_t k = c0; __any(on && k < c1); k += G) {
            const int32_t t = on && k + gl < c1 ? rsnap[k + gl] : -1;
            if (t >= 0) {
                lo = min(lo, t);
                hi = max(hi, t);
            }
        }
        const int32_t root = group_min<G>(lo);
        bool mixed = group_max<G>(hi) > root;
        group_boxes<G>(on && root != INT_MAX && !mixed, r0, r1, r0, -1, rboxes, c1, INT_MAX,
                       [&](bool valid, int32_t b2) {
            const int32_t t = valid ? rsnap[b2] : -1;
            const bool other = (ballot(t >= 0 && t != root) & gmask) != 0;
            mixed = mixed || other;
            return other;
        });
        mixed = mixed && on && root != INT_MAX;
        for (int32_t k = c0; __any(mixed && k < c1); k += G) {
            const bool put = mixed && k + gl < c1 && rsnap[k + gl] >= 0;
            const uint64_t puts = ballot(put);
            const unsigned int add = static_cast<unsigned int>(__popcll(puts));
            if (fill + add > kMixedStage) {
                unsigned int at = 0;
                if (lane_id() == 0) at = atomicAdd(count, fill);
                at = static_cast<unsigned int>(bcast(static_cast<int32_t>(at), 0));
                wave_lds_fence();
                for (unsigned int e = lane_id(); e < fill; e += kWave) list[at + e] = stage[w][e];
                wave_lds_fence();
                fill = 0;
            }
            if (put) stage[w][fill + __popcll(puts & lanemask_lt())] = k + gl;
            fill += add;
        }
    }
    // the rest, one reservation per block
    if (lane_id() == 0) left[w] = fill;
    __syncthreads();
    if (threadIdx.x == 0) {
        unsigned int sum = 0;
        for (int k = 0; k < kWavesPerBlock; ++k) sum += left[k];
        at0 = sum > 0 ? atomicAdd(count, sum) : 0u;
    }
    __syncthreads();
    unsigned int at = at0;
    for (int k = 0; k < w; ++k) at += left[k];
    for (unsigned int e = lane_id(); e < fill; e += kWave) list[at + e] = stage[w][e];
}

// The exact union: every listed box meets the later boxes of its
// neighbourhood that are in another snapshot tree (rsnap) and within eps
// (bounding boxes) -- the open pairs, counted in *nopen.  A pair is skipped
// when the two boxes are joined by now (live roots); two boxes wholly within
// eps of each other join at once; small pairs are tested by their lane; a
// pair with a box of more than kHeavyRows rows leaves an entry per kHeavyRows
// of that box in heavy (up to heavy_cap entries; beyond, the wave tests it
// here) and the others are tested by the wave.

// (Float rows up to 3-D: 5 waves per SIMD instead of 4, 4096 clouds of 8k rows
// 2.04 -> 1.75 ms; 6 waves 2.2.  The hook forest spills at 5: 2.8 -> 4.8 ms.)
template <typename T, int D>
__global__ __launch_bounds__(kThreads, D <= 3 && sizeof(T) == 4 ? 5 : 1) void k_box_union(
    const BoxArgs<T> a, const uint32_t* __restrict__ roff, const int2* __restrict__ rboxes,
    const int32_t* __restrict__ rsnap, const uint8_t* __restrict__ core,
    const int32_t* __restrict__ blist, const unsigned int* __restrict__ nlist_dev,
    int32_t* bparent, int2* __restrict__ heavy, unsigned long long* __restrict__ nheavy,
    unsigned long long heavy_cap, unsigned long long* __restrict__ nopen) {
    constexpr int G = kPairGroup<D>;
    constexpr int kPer = 64 / G;
    const int32_t nlist = uniform(static_cast<int32_t>(*nlist_dev));
    const int grp = lane_id() / G;
    const Span<T>* bbox = static_cast<const Span<T>*>(a.bbox);
    unsigned long long opened = 0;
    for (int32_t base = first_wave() * kPer; base < nlist; base += wave_stride() * kPer) {
        const bool on = base + grp < nlist;
        const int32_t b = blist[on ? base + grp : nlist - 1];
        const int32_t s0 = a.bstart[b], s1 = a.bstart[b + 1];
        const int32_t sb = rsnap[b];
        const int32_t u = a.bcell[b];
        const JobParams<T>& jp = a.jobs[a.njobs == 1 ? 0 : a.job_of_cell[u]];
        const T eps2 = jp.eps2;
        Span<T> mine[D];
#pragma unroll
        for (int j = 0; j < D; ++j) mine[j] = bbox[static_cast<int64_t>(b) * D + j];
        const int32_t r0 = static_cast<int32_t>(roff[u]);
        group_boxes<G>(on, r0, static_cast<int32_t>(roff[u + 1]), r0, -1, rboxes, b + 1, INT_MAX,
                       [&](bool valid, int32_t b2) {
            const int32_t s2 = valid ? rsnap[b2] : -1;
            bool open = false, whole = false;
            if (s2 >= 0 && s2 != sb) {
                T gap2, far2;
                box_gap<T, D>(bbox, b2, mine, gap2, far2);
                open = gap2 <= eps2;
                whole = far2 <= eps2;
                opened += open ? 1 : 0;
            }
            if (!__any(open)) return false;
            int32_t q0 = 0, q1 = 0;
            if (open) {
                const int32_t r = uf_find(bparent, sb), r2 = uf_find(bparent, s2);
                open = r != r2;
                if (open) {
                    q0 = a.bstart[b2];
                    q1 = a.bstart[b2 + 1];
                    const int64_t tests = static_cast<int64_t>(s1 - s0) * (q1 - q0);
                    if (whole || tests <= kLanePair) {
                        if (whole || lane_pair<T, D>(a.soa, a.ld, core, s0, s1, q0, q1, eps2))
                            uf_unite(bparent, r, r2);
                        open = false;
                    }
                }
            }
            for (uint64_t todo = ballot(open); todo != 0; todo &= todo - 1) {
                const int j = static_cast<int>(__builtin_ctzll(todo));
                const int32_t bj = bcast(b, j), b2j = bcast(b2, j);
                const int32_t r = uniform(uf_find(bparent, bj));
                const int32_t r2 = uniform(uf_find(bparent, b2j));
                if (r == r2) continue;
                const int32_t t0 = bcast(s0, j), t1 = bcast(s1, j);
                const int32_t v0 = bcast(q0, j), v1 = bcast(q1, j);
                if (max(t1 - t0, v1 - v0) > kHeavyRows) {
                    // the larger box by parts, each against the other box
                    const bool mine = t1 - t0 >= v1 - v0;
                    const int32_t x0 = mine ? t0 : v0, x1 = mine ? t1 : v1;
                    const int32_t k = (x1 - x0 + kHeavyRows - 1) / kHeavyRows;
                    unsigned long long at = 0;
                    if (lane_id() == 0) at = atomicAdd(nheavy, static_cast<unsigned long long>(k));
                    at = bcast64(at, 0);
                    const bool fits = at + static_cast<unsigned long long>(k) <= heavy_cap;
                    // (the entries of a range that does not fit do nothing)
                    for (int32_t e = lane_id(); e < k && at + e < heavy_cap; e += kWave)
                        heavy[at + e] = fits ? make_int2(x0 + e * kHeavyRows, mine ? b2j : bj)
                                             : make_int2(-1, -1);
                    if (fits) continue;
                }
                if (wave_pair<T, D>(a.soa, a.ld, core, bbox, t0, t1, b2j, v0, v1, bcast(eps2, j)) &&
                    lane_id() == 0)
                    uf_unite(bparent, r, r2);
            }
            return false;
        });
    }
    block_add<kThreads>(opened, nopen);
}

// The heavy entries (first slot of a part of a box, other box), one wave
// each: the part's core rows against the other box, unless the two are
// joined by now (looked at again every 64 rows).
template <typename T, int D>
__global__ __launch_bounds__(kThreads) void k_box_union_heavy(
    const BoxArgs<T> a, const int32_t* __restrict__ box_of_slot, const uint8_t* __restrict__ core,
    int32_t* bparent, const int2* __restrict__ heavy,
    const unsigned long long* __restrict__ nheavy, unsigned long long heavy_cap) {
    const unsigned long long found = *nheavy;
    const int32_t n = uniform(static_cast<int32_t>(found < heavy_cap ? found : heavy_cap));
    const Span<T>* bbox = static_cast<const Span<T>*>(a.bbox);
    for (int32_t w = first_wave(); w < n; w += wave_stride()) {
        const int32_t x0 = uniform(heavy[w].x), b2 = uniform(heavy[w].y);
        if (x0 < 0) continue;
        const int32_t b = uniform(box_of_slot[x0]);
        const int32_t x1 = min(uniform(a.bstart[b + 1]), x0 + kHeavyRows);
        const int32_t q0 = uniform(a.bstart[b2]), q1 = uniform(a.bstart[b2 + 1]);
        const JobParams<T>& jp = a.jobs[uniform(a.job_of_cell[uniform(a.bcell[b])])];
        for (int32_t c = x0; c < x1; c += kWave) {
            const int32_t r = uniform(uf_find(bparent, b));
            const int32_t r2 = uniform(uf_find(bparent, b2));
            if (r == r2) break;
            if (wave_pair<T, D>(a.soa, a.ld, core, bbox, c, min(c + kWave, x1), b2, q0, q1,
                                jp.eps2)) {
                if (lane_id() == 0) uf_unite(bparent, r, r2);
                break;
            }
        }
    }
}

// list[...] = every box with cores (v = bmincore != INT_MAX); *count +=
// their number; every box a root of its own (bparent), its smallest core key
// (cmin) none yet
__global__ __launch_bounds__(kThreads) void k_list_boxes(Count nbox_c,
                                                         const int32_t* __restrict__ bmincore,
                                                         int32_t* __restrict__ list,
                                                         unsigned int* __restrict__ count,
                                                         int32_t* __restrict__ bparent,
                                                         unsigned long long* __restrict__ cmin) {
    block_collect(nbox_c.get(), list, count, [&](int64_t b, int32_t& v) {
        v = static_cast<int32_t>(b);
        bparent[b] = v;
        cmin[b] = ~0ull;
        return bmincore[b] != INT_MAX;
    });
}

__global__ __launch_bounds__(kThreads) void k_core_init(
    int64_t n, const int32_t* __restrict__ box_of_slot, const uint8_t* __restrict__ btight,
    const int32_t* __restrict__ bstart, const int32_t* __restrict__ bcell,
    const uint32_t* __restrict__ inrow, uint8_t* __restrict__ core, int32_t* __restrict__ bmincore,
    int2* __restrict__ rows, unsigned int* __restrict__ nrows, int chunk) {
    block_collect(n, rows, nrows, [&](int64_t s, int2& v) {
        const int32_t b = box_of_slot[s];
        const uint8_t t = btight[b];
        const bool full = (t & 2) != 0;
        core[s] = full ? 1 : 0;
        const int32_t at = static_cast<int32_t>(s) - bstart[b];
        if (at == 0) bmincore[b] = full ? static_cast<int32_t>(inrow[s]) : INT_MAX;
        if (full || !(t & 4) || (at & (chunk - 1)) != 0) return false;
        v = make_int2(static_cast<int32_t>(s), bcell[b]);
        return true;
    });
}

// root of every box's tree -> rsnap (-1 for boxes without cores); with a
// list, the roots go there (*count += their number).  A hook leads to a box at
// most a cell away, so a tree is as deep as its cluster is wide, mostly along
// runs of consecutive boxes: the chains inside a block's tile of boxes are
// first shortened in LDS (jumps that double), so that the loads from memory
// that depend on each other are one per tile passed (300k 2-D rows, both
// rounds: 81 -> 18 us).  Every box ends up pointing at its root.
__global__ __launch_bounds__(kThreads) void k_box_roots(Count nbox_c,
                                                        const int32_t* __restrict__ bmincore,
                                                        int32_t* bparent,
                                                        int32_t* __restrict__ rsnap,
                                                        int32_t* __restrict__ list,
                                                        unsigned int* __restrict__ count) {
    __shared__ int32_t up[kCollectTile];
    const int64_t nbox = nbox_c.get();
    for (int64_t t = static_cast<int64_t>(blockIdx.x) * kCollectTile; t < nbox;
         t += static_cast<int64_t>(gridDim.x) * kCollectTile) {
        const int32_t t0 = static_cast<int32_t>(t);
        const int32_t len = static_cast<int32_t>(min(nbox - t, static_cast<int64_t>(kCollectTile)));
        int32_t p[kCollectPer];
#pragma unroll
        for (int k = 0; k < kCollectPer; ++k) {
            const int32_t e = static_cast<int32_t>(threadIdx.x) + k * kThreads;
            p[k] = e < len ? bparent[t0 + e] : -1;
            up[e] = p[k];
        }
        __syncthreads();
        bool more = true;
        for (int round = 0; more && round < 32; ++round) {
            bool moved = false;
#pragma unroll
            for (int k = 0; k < kCollectPer; ++k) {
                const int32_t q = p[k] >= t0 ? up[p[k] - t0] : p[k];
                moved = moved || q != p[k];
                p[k] = q;
            }
            more = __syncthreads_or(moved ? 1 : 0) != 0;  // (all have read)
#pragma unroll
            for (int k = 0; k < kCollectPer; ++k)
                up[static_cast<int32_t>(threadIdx.x) + k * kThreads] = p[k];
            __syncthreads();
        }
#pragma unroll
        for (int k = 0; k < kCollectPer; ++k) {
            const int32_t e = static_cast<int32_t>(threadIdx.x) + k * kThreads;
            if (e < len && p[k] != t0 + e) st_agent(&bparent[t0 + e], p[k]);
        }
    }
    __syncthreads();
    block_collect(nbox, list, count, [&](int64_t i, int32_t& v) {
        const int32_t b = static_cast<int32_t>(i);
        const int32_t r = bmincore[b] == INT_MAX ? -1 : uf_find(bparent, b);
        rsnap[b] = r;
        if (r >= 0 && r != b) st_agent(&bparent[b], r);
        v = b;
        return list && r == b;
    });
}

// Cluster ids.  A sorted position orders rows by (occupied cell, input
// row), so the smallest position of a component's cores is the smallest
// key (cell << 32 | row) of its boxes' smallest core rows (bmincore holds
// the input row); the position itself is the cell's first slot plus the
// number of the cell's rows with a smaller input row (every box of the
// cell holds its rows in input order, so a binary search per box counts).
__global__ __launch_bounds__(kThreads) void k_box_compmin(Count nbox_c,
                                                          const int32_t* __restrict__ bmincore,
                                                          const int32_t* __restrict__ bcell,
                                                          int32_t* bparent,
                                                          unsigned long long* __restrict__ cmin) {
    const int32_t nbox = static_cast<int32_t>(nbox_c.get());
    const int32_t b = static_cast<int32_t>(blockIdx.x) * kThreads + threadIdx.x;
    const bool act = b < nbox && bmincore[b] != INT_MAX;
    // neighbouring boxes mostly share their root: lanes of a run of equal
    // roots combine first, and only the run's first lane takes the atomic
    const int32_t r = act ? uf_find(bparent, b) : -1 - lane_id();
    unsigned long long key = act ? (static_cast<unsigned long long>(bcell[b]) << 32) |
                                       static_cast<uint32_t>(bmincore[b])
                                 : ~0ull;
    key = run_suffix_min<unsigned long long>(key, r);
    const bool head = run_head(r);  // every lane takes part in the shuffles
    if (act && head) atomicMin(&cmin[r], key);
}

// number of entries < row in the ascending v[lo, hi)
__device__ __forceinline__ int32_t count_below(const uint32_t* __restrict__ v, int32_t lo,
                                               int32_t hi, uint32_t row) {
    const int32_t first = lo;
    while (lo < hi) {
        const int32_t mid = (lo + hi) >> 1;
        if (v[mid] < row) lo = mid + 1;
        else hi = mid;
    }
    return lo - first;
}

// position of every component root's smallest core, one thread per box
// (non-roots leave at once)
__global__ __launch_bounds__(kThreads) void k_box_resolve(
    Count nbox_c, const int32_t* __restrict__ bparent, const unsigned long long* __restrict__ cmin,
    const int32_t* __restrict__ cbox, const int32_t* __restrict__ bstart,
    const uint32_t* __restrict__ inrow, const int32_t* __restrict__ ustart,
    int32_t* __restrict__ pos) {
    const int32_t nbox = static_cast<int32_t>(nbox_c.get());
    const int32_t r = static_cast<int32_t>(blockIdx.x) * kThreads + threadIdx.x;
    if (r >= nbox || bparent[r] != r) return;
    const unsigned long long key = cmin[r];
    if (key == ~0ull) return;  // no cores
    const int32_t u = static_cast<int32_t>(key >> 32);
    const uint32_t row = static_cast<uint32_t>(key & 0xffffffffu);
    int32_t below = 0;
    for (int32_t b2 = cbox[u]; b2 < cbox[u + 1]; ++b2)
        below += count_below(inrow, bstart[b2], bstart[b2 + 1], row);
    pos[r] = ustart[u] + below;
}

// cluster id (smallest core position of the component) per box with cores
__global__ __launch_bounds__(kThreads) void k_box_cluster(Count nbox_c,
                                                          const int32_t* __restrict__ bmincore,
                                                          int32_t* bparent,
                                                          const int32_t* __restrict__ compmin,
                                                          int32_t* __restrict__ bcluster) {
    const int32_t nbox = static_cast<int32_t>(nbox_c.get());
    const int32_t b = static_cast<int32_t>(blockIdx.x) * kThreads + threadIdx.x;
    if (b >= nbox) return;
    bcluster[b] = bmincore[b] == INT_MAX ? -1 : compmin[uf_find(bparent, b)];
}

// 16 bytes per store, then the rest
__global__ __launch_bounds__(kThreads) void k_fill_i32(int32_t* __restrict__ a, int32_t v,
                                                       int64_t n) {
    const int64_t n4 = n / 4;
    const int64_t stride = static_cast<int64_t>(gridDim.x) * kThreads;
    const int64_t i0 = static_cast<int64_t>(blockIdx.x) * kThreads + threadIdx.x;
    for (int64_t i = i0; i < n4; i += stride) reinterpret_cast<int4*>(a)[i] = make_int4(v, v, v, v);
    if (i0 < n - 4 * n4) a[4 * n4 + i0] = v;
}

}  // namespace

int box_split(int d) { return d <= 3 ? 2 : 3; }

int box_sub_bits(int d) { return box_sub_bits(d, box_split(d)); }

int box_sub_bits(int d, int k) {
    uint64_t v = 1;
    for (int j = 0; j < d; ++j) v *= static_cast<uint64_t>(k);
    const uint64_t mx = v - 1;
    return mx == 0 ? 0 : 64 - __builtin_clzll(mx);
}


template <typename T, int D>
void launch_gather_boxes(const T* pts, int64_t n, const uint32_t* inrow_of_slot, T* soa,
                         int64_t ld, const int32_t* box_of_slot, const int32_t* bstart, void* bbox,
                         void* part, hipStream_t s) {
    using U = OrdKey<T>;
    if (n <= 0) return;
    int64_t tile = kThreads;
    if constexpr (D * sizeof(T) <= 8) {
        if (!pts) tile = kBoundsTile;  // coordinates in place: bounding boxes only
    }
    const int64_t nb = (n + tile - 1) / tile;
    if (tile == kThreads) {
        hipLaunchKernelGGL((k_gather_boxes<T, D>), dim3(static_cast<unsigned>(nb)), dim3(kThreads),
                           0, s, pts, n, inrow_of_slot, soa, ld, box_of_slot, bstart,
                           static_cast<Span<T>*>(bbox), static_cast<U*>(part));
    } else {
        if constexpr (D * sizeof(T) <= 8)
            hipLaunchKernelGGL((k_box_bounds<T, D>), dim3(static_cast<unsigned>(nb)),
                               dim3(kThreads), 0, s, soa, ld, n, box_of_slot, bstart,
                               static_cast<Span<T>*>(bbox), static_cast<U*>(part));
    }
    hipLaunchKernelGGL((k_box_span<T, D>), dim3(blocks_for(nb, kWavesPerBlock)), dim3(kThreads), 0,
                       s, n, nb, tile, box_of_slot, bstart, static_cast<const U*>(part),
                       static_cast<Span<T>*>(bbox));
    HPD_HIP(hipGetLastError());
}

size_t gather_part_bytes(int64_t n, int d, int value_bytes) {
    const size_t nb = static_cast<size_t>((n + kThreads - 1) / kThreads);
    return 2 * nb * 2 * static_cast<size_t>(d) * static_cast<size_t>(value_bytes);
}

template <typename K>
void launch_box_table(const K* keys, int64_t n, int shift, uint32_t* sums, int32_t* box_of_slot,
                      int32_t* bstart, int32_t* bcell, K* ucell, int32_t* ustart, int32_t* cbox,
                      int32_t* ctab, uint32_t* nbox_dev, uint32_t* ncells_dev, hipStream_t s) {
    if (n <= 0) return;
    const int run = table_run(n);
    const dim3 grid(static_cast<unsigned>((table_tiles(n) + run - 1) / run));
    uint2* part = reinterpret_cast<uint2*>(sums);
    hipLaunchKernelGGL(k_table_count<K>, grid, dim3(kThreads), 0, s, keys, n, shift, run, part);
    hipLaunchKernelGGL(k_table_write<K>, grid, dim3(kThreads), 0, s, keys, n, shift, run,
                       static_cast<const uint2*>(part), box_of_slot, bstart, bcell, ucell, ustart,
                       cbox, ctab, nbox_dev, ncells_dev);
    HPD_HIP(hipGetLastError());
}

template <typename T, int D>
void launch_box_tight(const BoxArgs<T>& a, const uint8_t* cell_core, uint8_t* btight,
                      unsigned int* nloose, int32_t large, unsigned int* nlarge, hipStream_t s) {
    using U = OrdKey<T>;
    if (a.nbox <= 0) return;
    hipLaunchKernelGGL((k_box_tight<T, D>), dim3(blocks_for(a.nbox, kThreads)), dim3(kThreads), 0,
                       s, static_cast<const Span<T>*>(a.bbox), Count{a.nbox, a.nbox_dev}, a.bstart,
                       a.bcell, a.job_of_cell, a.jobs, cell_core, btight, nloose, large, nlarge);
}

void launch_list_boxes(Count nbox, const int32_t* bmincore, int32_t* list, unsigned int* count,
                       int32_t* bparent, unsigned long long* cmin, hipStream_t s) {
    if (nbox.host <= 0) return;
    hipLaunchKernelGGL(k_list_boxes, dim3(collect_blocks(nbox.host)), dim3(kThreads), 0, s, nbox,
                       bmincore, list, count, bparent, cmin);
    HPD_HIP(hipGetLastError());
}

template <typename T, int D>
void launch_box_hook(const BoxArgs<T>& a, const uint32_t* roff, const int2* rboxes,
                     const int32_t* bmincore, const uint8_t* core, const int32_t* blist,
                     const unsigned int* nlist, int32_t* bparent, hipStream_t s) {
    if (a.nbox <= 0) return;
    hipLaunchKernelGGL((k_box_link<T, D, false>),
                       dim3(persistent_blocks<k_box_link<T, D, false>>(a.nbox, 64 / kPairGroup<D>)),
                       dim3(kThreads), 0, s, a, roff, rboxes, bmincore, core, blist, nlist, bparent);
    HPD_HIP(hipGetLastError());
}

void launch_box_roots(Count nbox, const int32_t* bmincore, int32_t* bparent, int32_t* rsnap,
                      int32_t* list, unsigned int* count, hipStream_t s) {
    if (nbox.host <= 0) return;
    hipLaunchKernelGGL(k_box_roots, dim3(collect_blocks(nbox.host)), dim3(kThreads), 0, s, nbox,
                       bmincore, bparent, rsnap, list, count);
    HPD_HIP(hipGetLastError());
}

template <typename T, int D>
void launch_box_root_join(const BoxArgs<T>& a, const uint32_t* roff, const int2* rboxes,
                          const int32_t* rsnap, const uint8_t* core, const int32_t* roots,
                          const unsigned int* nroots, int32_t* bparent, hipStream_t s) {
    if (a.nbox <= 0) return;
    hipLaunchKernelGGL((k_box_link<T, D, true>),
                       dim3(persistent_blocks<k_box_link<T, D, true>>(a.nbox, 64 / kPairGroup<D>)),
                       dim3(kThreads), 0, s, a, roff, rboxes, rsnap, core, roots, nroots, bparent);
    HPD_HIP(hipGetLastError());
}

void launch_core_init(int64_t n, const int32_t* box_of_slot, const uint8_t* btight,
                      const int32_t* bstart, const int32_t* bcell, const uint32_t* inrow,
                      uint8_t* core, int32_t* bmincore, int2* rows, unsigned int* nrows,
                      int chunk, hipStream_t s) {
    if (n <= 0) return;
    hipLaunchKernelGGL(k_core_init, dim3(collect_blocks(n)), dim3(kCollectThreads), 0, s, n,
                       box_of_slot, btight, bstart, bcell, inrow, core, bmincore, rows, nrows, chunk);
    HPD_HIP(hipGetLastError());
}

template <typename T, int D>
void launch_box_union(const BoxArgs<T>& a, const uint32_t* roff, const int2* rboxes,
                      const int32_t* rsnap, const uint8_t* core, const int32_t* blist,
                      const unsigned int* nblist, Count m, int32_t* list, unsigned int* nlist,
                      const int32_t* box_of_slot, int2* heavy,
                      unsigned long long* nheavy, unsigned long long heavy_cap, int32_t* bparent,
                      unsigned long long* nopen, bool large, hipStream_t s) {
    if (a.nbox <= 0) return;
    // (a device-written number of boxes: the bound is the rows)
    const int64_t boxes = a.nbox_dev ? a.nbox / 8 : a.nbox;
    if (D >= 4 || boxes > kMixedBoxes) {
        hipLaunchKernelGGL(k_mixed_cells<D>,
                           dim3(persistent_blocks<k_mixed_cells<D>>(m.host, 64 / kPairGroup<D>)),
                           dim3(kThreads), 0, s, m, a.cbox, roff, rboxes, rsnap, list, nlist);
        blist = list;
        nblist = nlist;
    }
    hipLaunchKernelGGL((k_box_union<T, D>),
                       dim3(persistent_blocks<k_box_union<T, D>>(a.nbox, 64 / kPairGroup<D>)),
                       dim3(kThreads), 0, s, a, roff, rboxes, rsnap, core, blist, nblist, bparent,
                       heavy, nheavy, heavy_cap, nopen);
    // (its waves leave at once when there are no entries)
    if (large)
        hipLaunchKernelGGL((k_box_union_heavy<T, D>),
                       dim3(persistent_blocks<k_box_union_heavy<T, D>>(a.nrows / kHeavyRows + 1, 1)),
                       dim3(kThreads), 0, s, a, box_of_slot, core, bparent, static_cast<const int2*>(heavy),
                       static_cast<const unsigned long long*>(nheavy), heavy_cap);
    HPD_HIP(hipGetLastError());
}

void fill_i32(int32_t* p, int32_t v, int64_t n, hipStream_t s) {
    if (n <= 0) return;
    if (reinterpret_cast<uintptr_t>(p) % 16 != 0) throw Error(HPD_EINVAL, "fill_i32: 16-byte alignment");
    hipLaunchKernelGGL(k_fill_i32, dim3(std::min(blocks_for(n / 4 + 1, kThreads), 4096u)),
                       dim3(kThreads), 0, s, p, v, n);
}

void launch_box_clusters(Count nbox, const int32_t* bmincore, const int32_t* bcell,
                         const int32_t* cbox, const int32_t* bstart, const uint32_t* inrow,
                         const int32_t* ustart, int32_t* bparent, unsigned long long* cmin,
                         int32_t* compmin, int32_t* bcluster, hipStream_t s) {
    if (nbox.host <= 0) return;
    const dim3 g(blocks_for(nbox.host, kThreads));
    hipLaunchKernelGGL(k_box_compmin, g, dim3(kThreads), 0, s, nbox, bmincore, bcell, bparent, cmin);
    hipLaunchKernelGGL(k_box_resolve, g, dim3(kThreads), 0, s, nbox,
                       static_cast<const int32_t*>(bparent),
                       static_cast<const unsigned long long*>(cmin), cbox, bstart, inrow, ustart,
                       compmin);
    hipLaunchKernelGGL(k_box_cluster, g, dim3(kThreads), 0, s, nbox, bmincore, bparent,
                       static_cast<const int32_t*>(compmin), bcluster);
}

// Sorted positions of all slots (for the slot-level union and the
// one-thread border rule): a stable sort of the slots by occupied cell in
// input order gives the (cell, input row) order.
__global__ __launch_bounds__(kThreads) void k_pos_keys(int64_t n, const int32_t* __restrict__ box_of_slot,
                                                       const int32_t* __restrict__ bcell,
                                                       const uint32_t* __restrict__ inrow,
                                                       uint32_t* __restrict__ keys,
                                                       uint32_t* __restrict__ vals) {
    const int64_t s = static_cast<int64_t>(blockIdx.x) * kThreads + threadIdx.x;
    if (s >= n) return;
    const uint32_t r = inrow[s];
    keys[r] = static_cast<uint32_t>(bcell[box_of_slot[s]]);
    vals[r] = static_cast<uint32_t>(s);
}

__global__ __launch_bounds__(kThreads) void k_pos_scatter(int64_t n,
                                                          const uint32_t* __restrict__ slot_at,
                                                          uint32_t* __restrict__ pos_of_slot) {
    const int64_t i = static_cast<int64_t>(blockIdx.x) * kThreads + threadIdx.x;
    if (i < n) pos_of_slot[slot_at[i]] = static_cast<uint32_t>(i);
}

void launch_positions(int64_t n, int32_t m, const int32_t* box_of_slot, const int32_t* bcell,
                      const uint32_t* inrow, uint32_t* keys_a, uint32_t* vals_a, uint32_t* keys_b,
                      uint32_t* vals_b, uint32_t* hist, uint32_t* tmp, uint32_t* pos_of_slot,
                      hipStream_t s) {
    if (n <= 0) return;
    hipLaunchKernelGGL(k_pos_keys, dim3(blocks_for(n, kThreads)), dim3(kThreads), 0, s, n,
                       box_of_slot, bcell, inrow, keys_a, vals_a);
    const int bits = m > 1 ? 64 - __builtin_clzll(static_cast<unsigned long long>(m - 1)) : 0;
    const bool in_b = radix_sort_pairs<uint32_t>(keys_a, vals_a, keys_b, vals_b, n, bits, hist, tmp, s);
    hipLaunchKernelGGL(k_pos_scatter, dim3(blocks_for(n, kThreads)), dim3(kThreads), 0, s, n,
                       static_cast<const uint32_t*>(in_b ? vals_b : vals_a), pos_of_slot);
    HPD_HIP(hipGetLastError());
}

#define HPD_INST_BOX_KEYS(T, D)                                                                   \
    template void launch_gather_boxes<T, D>(const T*, int64_t, const uint32_t*, T*, int64_t,      \
                                            const int32_t*, const int32_t*, void*, void*,         \
                                            hipStream_t);                                         \
    template void launch_box_tight<T, D>(const BoxArgs<T>&, const uint8_t*, uint8_t*,            \
                                         unsigned int*, int32_t, unsigned int*,           \
                                         hipStream_t);                                            \
    template void launch_box_hook<T, D>(const BoxArgs<T>&, const uint32_t*, const int2*,          \
                                        const int32_t*, const uint8_t*, const int32_t*,           \
                                        const unsigned int*, int32_t*, hipStream_t);              \
    template void launch_box_root_join<T, D>(const BoxArgs<T>&, const uint32_t*, const int2*,     \
                                             const int32_t*, const uint8_t*, const int32_t*,      \
                                             const unsigned int*, int32_t*, hipStream_t);         \
    template void launch_box_union<T, D>(const BoxArgs<T>&, const uint32_t*, const int2*,         \
                                         const int32_t*, const uint8_t*, const int32_t*,          \
                                         const unsigned int*, Count, int32_t*, unsigned int*,     \
                                         const int32_t*, int2*,                                   \
                                         unsigned long long*, unsigned long long, int32_t*,       \
                                         unsigned long long*, bool, hipStream_t);
#define HPD_INST_BOX_ALL_D(T) \
    HPD_INST_BOX_KEYS(T, 1)   \
    HPD_INST_BOX_KEYS(T, 2)   \
    HPD_INST_BOX_KEYS(T, 3)   \
    HPD_INST_BOX_KEYS(T, 4)   \
    HPD_INST_BOX_KEYS(T, 5)   \
    HPD_INST_BOX_KEYS(T, 6)   \
    HPD_INST_BOX_KEYS(T, 7)   \
    HPD_INST_BOX_KEYS(T, 8)
HPD_INST_BOX_ALL_D(float)
HPD_INST_BOX_ALL_D(double)

#define HPD_INST_BOX_TABLE(K)                                                              \
    template void launch_box_table<K>(const K*, int64_t, int, uint32_t*, int32_t*, int32_t*, \
                                      int32_t*, K*, int32_t*, int32_t*, int32_t*, uint32_t*, \
                                      uint32_t*, hipStream_t);
HPD_INST_BOX_TABLE(uint32_t)
HPD_INST_BOX_TABLE(uint64_t)

}  // namespace hpd
