// Neighbour-cell kernels of the clustering pass.
//
// Replaces local_dbscan (hpdbscan.h:51-101), region_query
// (spatial_index.h:739-768), the rules merge (rules.h, hpdbscan.h:198-211)
// and the scatter back to input order (spatial_index.h:852-872).
//
// The result the reference computes is order independent except for one
// case (border rows next to cores of two clusters):
//   core(p)  <=>  |{q in candidates(p) : dist2(p, q) <= EPS2}| >= minPts
//   cluster of a core = 1 + smallest sorted position of a core in its
//                       eps-connected component of cores
//   border row: within eps of a core; noise: neither.
// The kernels compute exactly that:
//   k_core    count within-eps candidates per row, stop at minPts
//   k_hook    every core points at the smallest adjacent core before it
//             (a forest whose roots are local minima; parent[x] <= x)
//   k_roots   root of every core (path-halving find), snapshot of the
//             roots, and per occupied cell the smallest / largest root of
//             its cores
//   k_union   union-find over the core pairs not yet known to be connected:
//             a neighbour row whose cells hold only cores of the chunk's
//             single root is skipped, a candidate whose snapshot root equals
//             the row's root is skipped, every other within-eps core pair
//             is united (larger root hooked under the smaller)
//   k_roots   final roots; core rows get -(root + 1)
//   k_border  smallest adjacent root for non-core rows (0 = noise); a
//             neighbourhood whose cells hold cores of one root only stops at
//             the first hit
// Each core pair is either tested or provably in one component already, so
// the components, and with them every label, are exact.
//
// Work decomposition: one wave per 64-row chunk of an occupied cell; lanes
// own the chunk's rows, the candidate rows stream through the wave in
// aligned batches fetched with wave-uniform addresses.
#include <algorithm>
#include <climits>
#include <type_traits>

#include "boxes.hpp"
#include "cellkey.hpp"
#include "collect.hpp"
#include "common.hpp"
#include "dbscan.hpp"
#include "grid.hpp"
#include "internal.hpp"
#include "put_off.hpp"
#include "visit.hpp"

namespace hpd {

namespace {

constexpr int kThreads = 256;
constexpr int kWavesPerBlock = kThreads / kWave;

// sorted position of a slot
__device__ __forceinline__ int32_t slot_pos(const uint32_t* __restrict__ pos_of_slot, int32_t s) {
    return pos_of_slot ? static_cast<int32_t>(pos_of_slot[s]) : s;
}

struct Chunk {
    int32_t u;       // occupied cell
    int32_t first;   // first row of the chunk
    int32_t end;     // end row of the cell
    int32_t r0, r1;  // its neighbour ranges (ascending, or nearest first)
};

__device__ __forceinline__ bool fetch_chunk(const int2* __restrict__ items, int32_t nitems,
                                            const int32_t* __restrict__ ustart,
                                            const uint32_t* __restrict__ roff, Chunk& c) {
    const int32_t wid = uniform(static_cast<int32_t>(blockIdx.x) * kWavesPerBlock +
                                static_cast<int32_t>(threadIdx.x >> 6));
    if (wid >= nitems) return false;
    const int2 it = items[wid];
    c.u = uniform(it.x);
    c.first = uniform(it.y);
    c.end = uniform(ustart[c.u + 1]);
    c.r0 = uniform(static_cast<int32_t>(roff[c.u]));
    c.r1 = uniform(static_cast<int32_t>(roff[c.u + 1]));
    return true;
}

__device__ __forceinline__ int32_t wave_min(int32_t v) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v = min(v, __shfl_xor(v, o, 64));
    return v;
}
__device__ __forceinline__ int32_t wave_max(int32_t v) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v = max(v, __shfl_xor(v, o, 64));
    return v;
}

// Every occupied cell in [a, b) holds either no core or only cores of root R.
__device__ __forceinline__ bool cells_single_root(int2 cs, const int32_t* __restrict__ cmin,
                                                  const int32_t* __restrict__ cmax, int32_t R) {
    for (int32_t c = cs.x; c < cs.y; ++c) {
        const int32_t mn = cmin[c], mx = cmax[c];
        if (mn <= mx && (mn != R || mx != R)) return false;
    }
    return true;
}

template <typename T, int D>
__global__ __launch_bounds__(kThreads) void k_core(const DbscanArgs<T> a, uint8_t* __restrict__ core,
                                                   unsigned long long* __restrict__ ncore) {
    Chunk c;
    if (!fetch_chunk(a.items, a.nitems, a.ustart, a.roff, c)) return;
    const JobParams<T>& jp = a.jobs[uniform(a.job_of_cell[c.u])];
    const T eps2 = jp.eps2;
    const uint32_t min_pts = jp.min_pts;
    const int32_t p = c.first + lane_id();
    const bool valid = p < c.end;
    T pc[D];
    load_row<T, D>(a.soa, a.ld, valid ? p : c.first, pc);
    uint32_t cnt = 0;
    // rows of a tight box with >= minPts rows are core without counting
    if (a.btight && valid && (a.btight[a.box_of_slot[p]] & 2)) cnt = min_pts;
    auto body = [&](int32_t, const T* qc, uint8_t, int32_t) {
        cnt += within<D>(pc, qc, eps2) ? 1u : 0u;
    };
    auto stop = [&] { return static_cast<bool>(__all(!valid || cnt >= min_pts)); };
    bool done = stop();
    // the cell's own row first: most neighbours are there
    const int32_t center = uniform(a.rcenter[c.u]);
    for (int32_t i = -1; i < c.r1 - c.r0 && !done; ++i) {
        const int32_t r = i < 0 ? center : c.r0 + i;
        if (i >= 0 && r == center) continue;
        const int2 rg = a.ranges[r];
        done = visit_range<T, D>(a.soa, a.ld, nullptr, nullptr, uniform(rg.x), uniform(rg.y), body,
                                 stop);
    }
    const bool is_core = valid && cnt >= min_pts;
    if (valid) core[p] = is_core ? 1 : 0;
    (void)ncore;
}

// Boxes of more rows are walked in parts of this many, one wave each
// (100M skewed rows: 26 us a part).
constexpr int32_t kHeavyWalk = 16384;

// An entry (slot, first row) per part of the rows [q0, q1) of a box; false
// when the list is full (every argument wave-uniform).
template <typename T>
__device__ __forceinline__ bool put_heavy(const DbscanArgs<T>& a, int32_t slot, int32_t q0,
                                          int32_t q1) {
    const int32_t k = (q1 - q0 + kHeavyWalk - 1) / kHeavyWalk;
    unsigned long long at = 0;
    if (lane_id() == 0) at = atomicAdd(a.nheavy, static_cast<unsigned long long>(k));
    at = bcast64(at, 0);
    const bool fits = at + static_cast<unsigned long long>(k) <= a.heavy_cap;
    // (the entries of a range that does not fit do nothing)
    for (int32_t e = lane_id(); e < k && at + e < a.heavy_cap; e += kWave)
        a.heavy[at + e] = fits ? make_int2(slot, q0 + e * kHeavyWalk) : make_int2(-1, -1);
    return fits;
}
template <typename T>
__device__ __forceinline__ int32_t heavy_count(const DbscanArgs<T>& a) {
    const unsigned long long n = *a.nheavy;
    return uniform(static_cast<int32_t>(n < a.heavy_cap ? n : a.heavy_cap));
}

// Box-mode core counts: the chunks listed in a.crows (up to G rows of one
// box, boxes outside the full ones, in cells that can hold cores), G lanes per
// chunk, a neighbour box per lane: the chunk's rows and counts lie in LDS, and
// each lane holds its box against one row after the other.  A box farther
// than eps from the row is skipped, one within eps of its farthest corner
// counts whole, the others are tested row by row: small ones by their lane,
// larger ones by the whole wave with the candidates on the lanes.
//
// Bound by VALU issue of the box tests and by the latency of list -> cell ->
// box ranges -> boxes, which the rows of a chunk share.  kCount: also add the
// row-row distance tests executed to *ntests (the instrumented variant).
// kHeavy: with a.heavy (boxes of more than kHeavyWalk rows exist) a row's walk
// of such a box leaves an entry per kHeavyWalk of its rows for k_core_heavy:
// one wave takes 0.4 us per 256 rows, 8 ms for a box of five million.  A
// variant of its own, since the code costs scalar registers (4096 clouds of 8k
// rows: 5.3 ms without, 9.0 ms with it).  Float rows up to 3-D fit 8 waves per
// SIMD (64 VGPRs, nothing spilled): the same clouds 5.35 ms at 7 waves, 4.95 at 8.
template <typename T, int D, bool kCount, bool kHeavy>
__global__ __launch_bounds__(kThreads, D <= 3 && sizeof(T) == 4 && !kCount ? 8 : 1)
void k_core_rows(const DbscanArgs<T> a, uint8_t* __restrict__ core,
                 unsigned long long* __restrict__ ntests) {
    constexpr int G = kGroup<D>;
    constexpr int kPer = 64 / G;  // chunks of a wave
    __shared__ T rows_lds[kWavesPerBlock][64][D];
    __shared__ uint32_t cnt_lds[kWavesPerBlock][64];
    const int w = static_cast<int>(threadIdx.x >> 6);
    const int32_t nitems = uniform(static_cast<int32_t>(*a.ncrows_dev));
    const int lane = lane_id();
    const int g0 = lane & ~(G - 1);  // first lane of the group
    T(*rx)[D] = rows_lds[w];
    uint32_t* rc = cnt_lds[w];
    // the lanes of the caller's group where `on`, as G bits
    auto group_bits = [&](bool on) {
        static_assert(G <= 32, "a group's lanes in 32 bits");
        return static_cast<uint32_t>(ballot(on) >> g0) & (~0u >> (32 - G));
    };
    const Span<T>* bbox = static_cast<const Span<T>*>(a.bbox);
    unsigned long long tests = 0;
    for (int32_t base = first_wave() * kPer; base < nitems; base += wave_stride() * kPer) {
        const int32_t i = base + lane / G;
        const bool on = i < nitems;
        const int2 it = a.crows[on ? i : nitems - 1];
        const int32_t u = it.y;
        const int32_t b = a.box_of_slot[it.x];
        const int32_t p = it.x + (lane & (G - 1));
        const bool has = on && p < a.bstart[b + 1];
        T pc[D];
        load_row<T, D>(a.soa, a.ld, has ? p : it.x, pc);
#pragma unroll
        for (int j = 0; j < D; ++j) rx[lane][j] = pc[j];
        rc[lane] = 0;
        wave_lds_fence();
        const int32_t r0 = static_cast<int32_t>(a.roff[u]);
        const int32_t r1 = static_cast<int32_t>(a.roff[u + 1]);
        const JobParams<T>& jp = a.jobs[a.njobs == 1 ? 0 : a.job_of_cell[u]];
        const T eps2 = jp.eps2;
        const uint32_t min_pts = jp.min_pts;
        bool need = has && min_pts > 0;
        bool put_off = false;  // the lane's row has entries in a.heavy
        group_boxes<G>(on && min_pts > 0, r0, r1, a.rcenter[u], a.cbox[u], a.rboxes, 0, INT_MAX,
                       [&](bool valid, int32_t b2) {
            int32_t q0 = 0, q1 = 0;
            uint32_t part = 0;  // rows of the chunk the box is undecided for
            const uint32_t open = group_bits(need);
            if (valid) {
                Span<T> s[D];
#pragma unroll
                for (int j = 0; j < D; ++j) s[j] = bbox[static_cast<int64_t>(b2) * D + j];
                q0 = a.bstart[b2];
                q1 = a.bstart[b2 + 1];
                for (uint32_t m = open; m != 0; m &= m - 1) {
                    const int k = __builtin_ctz(m);
                    T gmin2, gmax2;
                    point_box<T, D>(s, 0, rx[g0 + k], gmin2, gmax2);
                    if (gmin2 > eps2) continue;
                    if (gmax2 <= eps2) atomicAdd(&rc[g0 + k], static_cast<uint32_t>(q1 - q0));
                    else part |= 1u << k;
                }
            }
            wave_lds_fence();
            need = need && rc[lane] < min_pts;
            if (__any(part != 0)) {
                const bool lane_walk = q1 - q0 <= kLaneRows;
                part &= group_bits(need);
                if (lane_walk) {
                    for (uint32_t m = part; m != 0; m &= m - 1) {
                        const int k = __builtin_ctz(m);
                        uint32_t c = 0;
                        for (int32_t q = q0; q < q1; ++q) {
                            T qc[D];
                            load_row<T, D>(a.soa, a.ld, q, qc);
                            c += within<D>(rx[g0 + k], qc, eps2) ? 1u : 0u;
                        }
                        if (c) atomicAdd(&rc[g0 + k], c);
                        if constexpr (kCount) tests += static_cast<unsigned long long>(q1 - q0);
                    }
                }
                for (uint64_t todo = ballot(part != 0 && !lane_walk); todo != 0; todo &= todo - 1) {
                    const int j = static_cast<int>(__builtin_ctzll(todo));
                    const uint32_t mp = static_cast<uint32_t>(bcast(static_cast<int32_t>(min_pts), j));
                    for (uint32_t m = static_cast<uint32_t>(bcast(static_cast<int32_t>(part), j));
                         m != 0; m &= m - 1) {
                        const int row = (j & ~(G - 1)) + __builtin_ctz(m);
                        wave_lds_fence();
                        const uint32_t now =
                            static_cast<uint32_t>(uniform(static_cast<int32_t>(rc[row])));
                        if (now >= mp) continue;  // an earlier box was enough
                        if constexpr (kHeavy)
                            if (a.heavy_cap > 0 && bcast(q1 - q0, j) > kHeavyWalk &&
                                put_heavy(a, bcast(p, row), bcast(q0, j), bcast(q1, j))) {
                                if (lane == row) put_off = true;
                                continue;
                            }
                        T pr[D];
#pragma unroll
                        for (int e = 0; e < D; ++e) pr[e] = bcast(pc[e], row);
                        uint32_t visited = 0;
                        const uint32_t got = wide_count<T, D>(a.soa, a.ld, nullptr, bcast(q0, j),
                                                              bcast(q1, j), pr, bcast(eps2, j),
                                                              mp - now, visited);
                        if (lane == 0) rc[row] = now + got;
                        if constexpr (kCount)
                            if (lane == 0) tests += visited;
                    }
                }
                wave_lds_fence();
                need = need && rc[lane] < min_pts;
            }
            return group_bits(need) == 0;
        });
        // (launch_core_init wrote 0 for every listed row)
        wave_lds_fence();
        const bool is_core = has && rc[lane] >= min_pts;
        if constexpr (kHeavy)
            if (put_off) a.slot_a[p] = static_cast<int32_t>(min(rc[lane], min_pts));
        if (is_core) core[p] = 1;
        const int32_t first =
            group_min<G>(is_core ? static_cast<int32_t>(a.inrow[p]) : INT_MAX);
        if (lane == g0 && first != INT_MAX) atomicMin(&a.bmincore[b], first);
        wave_lds_fence();
    }
    if constexpr (kCount) block_add<kThreads>(tests, ntests);
}

// The put-off walks of k_core_rows, a wave per entry (slot, first row of the
// part): the counts meet in a.slot_a, and the part that brings a row to minPts
// makes it a core.
template <typename T, int D>
__global__ __launch_bounds__(kThreads) void k_core_heavy(const DbscanArgs<T> a,
                                                         uint8_t* __restrict__ core,
                                                         unsigned long long* __restrict__ ntests) {
    const int32_t n = heavy_count(a);
    unsigned long long tests = 0;
    for (int32_t w = first_wave(); w < n; w += wave_stride()) {
        const int32_t p = uniform(a.heavy[w].x), q0 = uniform(a.heavy[w].y);
        if (p < 0) continue;
        const int32_t b = uniform(a.box_of_slot[p]);
        const JobParams<T>& jp = a.jobs[uniform(a.job_of_cell[uniform(a.bcell[b])])];
        const uint32_t min_pts = jp.min_pts;
        const uint32_t now = static_cast<uint32_t>(uniform(ld_agent(&a.slot_a[p])));
        if (now >= min_pts) continue;
        const int32_t q1 = min(q0 + kHeavyWalk, uniform(a.bstart[uniform(a.box_of_slot[q0]) + 1]));
        T pc[D];
        load_row<T, D>(a.soa, a.ld, p, pc);
        uint32_t visited = 0;
        const uint32_t got = wide_count<T, D>(a.soa, a.ld, nullptr, q0, q1, pc, jp.eps2,
                                              min_pts - now, visited);
        if (lane_id() == 0) {
            tests += visited;
            if (got > 0) {
                const uint32_t old = static_cast<uint32_t>(
                    atomicAdd(&a.slot_a[p], static_cast<int32_t>(got)));
                if (old < min_pts && old + got >= min_pts) {
                    core[p] = 1;
                    atomicMin(&a.bmincore[b], static_cast<int32_t>(a.inrow[p]));
                }
            }
        }
    }
    if (ntests) block_add<kThreads>(tests, ntests);
}

template <typename T, int D>
__global__ __launch_bounds__(kThreads) void k_hook(const DbscanArgs<T> a,
                                                   const uint8_t* __restrict__ core,
                                                   int32_t* __restrict__ parent) {
    Chunk c;
    if (!fetch_chunk(a.items, a.nitems, a.ustart, a.roff, c)) return;
    const T eps2 = a.jobs[uniform(a.job_of_cell[c.u])].eps2;
    const int32_t p = c.first + lane_id();
    const bool valid = p < c.end;
    const bool active = valid && core[p];
    if (!__any(active)) return;
    T pc[D];
    load_row<T, D>(a.soa, a.ld, valid ? p : c.first, pc);
    // any within-eps core before p is a valid parent (parent[x] < x keeps the
    // hooks a forest); the first one found is taken
    int32_t best = p;
    bool found = !active;
    auto body = [&](int32_t q, const T* qc, uint8_t cq, int32_t) {
        if (!cq) return;
        if (!found && q < p && within<D>(pc, qc, eps2)) {
            best = q;
            found = true;
        }
    };
    auto stop = [&] { return static_cast<bool>(__all(found)); };
    const int32_t pmax = uniform(min(c.first + kWave, c.end) - 1);
    // a cell's rows may be stored nearest first rather than ascending, so a
    // row that starts at or after pmax is skipped, not taken as the end
    for (int32_t r = c.r0; r < c.r1; ++r) {
        const int2 rg = a.ranges[r];
        const int32_t qb = uniform(rg.x);
        if (qb >= pmax) continue;
        if (visit_range<T, D>(a.soa, a.ld, core, nullptr, qb, uniform(min(rg.y, pmax)), body, stop))
            break;
    }
    if (active) parent[p] = best;
}

// Roots of the chunk's cores (path-halving find), stored back into parent,
// snapshot copy, and per-cell smallest / largest root.
__global__ __launch_bounds__(kThreads) void k_roots(const int2* __restrict__ items, int32_t nitems,
                                                    const int32_t* __restrict__ ustart,
                                                    const uint32_t* __restrict__ roff,
                                                    const uint8_t* __restrict__ core,
                                                    int32_t* parent, int32_t* __restrict__ rsnap,
                                                    int32_t* __restrict__ cmin,
                                                    int32_t* __restrict__ cmax) {
    Chunk c;
    if (!fetch_chunk(items, nitems, ustart, roff, c)) return;
    const int32_t p = c.first + lane_id();
    const bool valid = p < c.end;
    const bool active = valid && core[p];
    if (!__any(active)) return;
    int32_t r = INT_MAX;
    if (active) {
        r = uf_find(parent, p);
        st_agent(&parent[p], r);
        rsnap[p] = r;
    }
    const int32_t rmin = wave_min(active ? r : INT_MAX);
    const int32_t rmax = wave_max(active ? r : -1);
    if (lane_id() == 0) {
        atomicMin(&cmin[c.u], rmin);
        atomicMax(&cmax[c.u], rmax);
    }
}

// smallest sorted position of every slot-level component
__global__ __launch_bounds__(kThreads) void k_compmin(const uint8_t* __restrict__ core,
                                                      int32_t* parent, int64_t n,
                                                      const uint32_t* __restrict__ pos_of_slot,
                                                      int32_t* __restrict__ compmin) {
    const int64_t i = static_cast<int64_t>(blockIdx.x) * kThreads + threadIdx.x;
    if (i >= n || !core[i]) return;
    const int32_t r = uf_find(parent, static_cast<int32_t>(i));
    const int32_t pos = pos_of_slot ? static_cast<int32_t>(pos_of_slot[i]) : static_cast<int32_t>(i);
    atomicMin(&compmin[r], pos);
}

// cluster of every core slot -> label, slot array of clusters, per-cell
// smallest / largest cluster
template <typename T>
__global__ __launch_bounds__(kThreads) void k_label_cores(
    const int2* __restrict__ items, int32_t nitems, const int32_t* __restrict__ ustart,
    const uint32_t* __restrict__ roff, const JobParams<T>* __restrict__ jobs,
    const int32_t* __restrict__ job_of_cell, const uint8_t* __restrict__ core,
    const int32_t* __restrict__ box_of_slot, const int32_t* __restrict__ bcluster, int32_t* parent,
    const int32_t* __restrict__ compmin, const uint32_t* __restrict__ inrow,
    int64_t* __restrict__ labels, int32_t* __restrict__ rootslot, int32_t* __restrict__ cmin,
    int32_t* __restrict__ cmax) {
    Chunk c;
    if (!fetch_chunk(items, nitems, ustart, roff, c)) return;
    const int32_t p = c.first + lane_id();
    const bool valid = p < c.end;
    const bool active = valid && core[p];
    if (!__any(active)) return;
    const int64_t first_pos = jobs[uniform(job_of_cell[c.u])].row_begin;
    int32_t r = INT_MAX;
    if (active) {
        r = bcluster ? bcluster[box_of_slot[p]] : compmin[uf_find(parent, p)];
        labels[inrow[p]] = -(static_cast<int64_t>(r) - first_pos + 1);
        rootslot[p] = r;
    }
    const int32_t rmin = wave_min(active ? r : INT_MAX);
    const int32_t rmax = wave_max(active ? r : -1);
    if (lane_id() == 0) {
        atomicMin(&cmin[c.u], rmin);
        atomicMax(&cmax[c.u], rmax);
    }
}

// Box mode: core labels one thread per slot (the cluster of a core is its
// box's); the other rows go to `rows` as (slot, cell) for k_border_rows.
// skip_full (with *full_ok set): the rows of full boxes (btight bit 2) were
// labelled in input order (k_label_full_rows) and are skipped here.
template <typename T>
__global__ __launch_bounds__(kThreads) void k_label_cores_boxes(
    int64_t n, const JobParams<T>* __restrict__ jobs, const int32_t* __restrict__ job_of_cell,
    const uint8_t* __restrict__ core, const int32_t* __restrict__ box_of_slot,
    const int32_t* __restrict__ bcell, const int32_t* __restrict__ bcluster,
    const uint32_t* __restrict__ inrow, int64_t* __restrict__ labels,
    int32_t* __restrict__ rootslot, unsigned long long* __restrict__ ncore, bool one_job,
    const uint8_t* __restrict__ skip_full, const unsigned int* __restrict__ full_ok,
    int2* __restrict__ rows, unsigned int* __restrict__ nrows) {
    if (skip_full && *full_ok == 0) skip_full = nullptr;
    unsigned long long cores = 0;  // of the run statistics
    block_collect(n, rows, nrows, [&](int64_t p, int2& v) {
        const int32_t b = box_of_slot[p];
        if (!core[p]) {
            v = make_int2(static_cast<int32_t>(p), bcell[b]);
            return true;
        }
        ++cores;  // every core, the row-order ones included
        if (skip_full && (skip_full[b] & 2)) return false;
        const int32_t r = bcluster[b];
        if (rootslot) rootslot[p] = r;
        // one job starts at row 0
        const int64_t first_pos = one_job ? 0 : jobs[job_of_cell[bcell[b]]].row_begin;
        labels[inrow[p]] = -(static_cast<int64_t>(r) - first_pos + 1);
        return false;
    });
    block_add<kThreads>(cores, ncore);
}

// Row-order labels of full boxes.  A table indexed by cell key (the sort's
// keys start at 0 and are dense enough when the largest one is below the
// table's capacity) holds, for the key of every full box (tight with >=
// minPts rows: every row core, cluster = the box's), the label's magnitude
// bcluster - first row of the job + 1, and 0 for the keys of other boxes.
// Keys no box has are never looked up.  *ok = the largest key fits.
template <typename T, typename K>
__global__ __launch_bounds__(kThreads) void k_full_box_table(
    const K* __restrict__ keys, int64_t n, const int32_t* __restrict__ bstart, Count nbox,
    const int32_t* __restrict__ bcell, const int32_t* __restrict__ job_of_cell,
    const JobParams<T>* __restrict__ jobs, const uint8_t* __restrict__ btight,
    const int32_t* __restrict__ bcluster, int32_t* __restrict__ tab, int64_t cap,
    unsigned int* __restrict__ ok) {
    const bool fits = static_cast<uint64_t>(keys[n - 1]) < static_cast<uint64_t>(cap);
    const int64_t b = static_cast<int64_t>(blockIdx.x) * kThreads + threadIdx.x;
    if (b == 0) *ok = fits ? 1u : 0u;
    if (!fits || b >= nbox.get()) return;
    int32_t v = 0;
    if (btight[b] & 2)
        v = static_cast<int32_t>(static_cast<int64_t>(bcluster[b]) -
                                 jobs[job_of_cell[bcell[b]]].row_begin + 1);
    tab[static_cast<int64_t>(keys[bstart[b]])] = v;
}

// The labels of the rows of full boxes, written in input order: each row's
// key is computed again from its coordinates exactly as the sort's keys
// were (row_key), looked up in the table, and the label stored at the row's
// own place (coalesced, where labelling in slot order stores at permuted
// places).  Rows of other boxes (table value 0) are left to
// k_label_cores_boxes.  Nothing when the table did not fit.
constexpr int kFullRows = 256;  // rows per wave
template <typename T, int D, typename K>
__global__ __launch_bounds__(kThreads) void k_label_full_rows(
    const T* __restrict__ pts, int64_t n, const JobParams<T>* __restrict__ jobs, int32_t njobs,
    int sub_k, int sub_bits, const int32_t* __restrict__ tab, int64_t cap,
    const unsigned int* __restrict__ ok, int64_t* __restrict__ labels) {
    if (*ok == 0) return;
    const int64_t r0 = (static_cast<int64_t>(blockIdx.x) * kWavesPerBlock + (threadIdx.x >> 6)) *
                       kFullRows;
    for_job_rows(jobs, njobs, r0, r0 + kFullRows < n ? r0 + kFullRows : n,
                 [&](const JobParams<T>& jp, int64_t i) {
        const K key = static_cast<K>(row_key<T, D>(pts + i * D, jp, sub_k, sub_bits));
        // (every row's key is a box's key, below cap when *ok is set)
        const int32_t v = static_cast<uint64_t>(key) < static_cast<uint64_t>(cap)
                              ? tab[static_cast<int64_t>(key)]
                              : 0;
        if (v != 0) labels[i] = -static_cast<int64_t>(v);
    });
}

template <typename T, int D>
__global__ __launch_bounds__(kThreads) void k_union(const DbscanArgs<T> a,
                                                    const uint8_t* __restrict__ core,
                                                    const int32_t* __restrict__ rsnap,
                                                    const int32_t* __restrict__ cmin,
                                                    const int32_t* __restrict__ cmax,
                                                    int32_t* parent) {
    Chunk c;
    if (!fetch_chunk(a.items, a.nitems, a.ustart, a.roff, c)) return;
    const T eps2 = a.jobs[uniform(a.job_of_cell[c.u])].eps2;
    const int32_t p = c.first + lane_id();
    const bool valid = p < c.end;
    const bool active = valid && core[p];
    if (!__any(active)) return;
    const int32_t rp = active ? rsnap[p] : -1;
    const int32_t rmin = wave_min(active ? rp : INT_MAX);
    const int32_t rmax = wave_max(active ? rp : -1);
    const int32_t R = uniform(rmin == rmax ? rmin : -1);  // the chunk's single root, if any
    T pc[D];
    load_row<T, D>(a.soa, a.ld, valid ? p : c.first, pc);
    // every core pair is handled by its larger position: only q < p
    const int32_t pmax = uniform(min(c.first + kWave, c.end) - 1);
    auto body = [&](int32_t q, const T* qc, uint8_t cq, int32_t rq) {
        if (!cq) return;
        const bool need = active && q < p && rq != rp;
        if (!__any(need)) return;
        if (need && within<D>(pc, qc, eps2)) uf_unite(parent, p, q);
    };
    auto never = [] { return false; };
    for (int32_t r = c.r0; r < c.r1; ++r) {
        const int2 rg = a.ranges[r];
        const int32_t qb = uniform(rg.x);
        if (qb >= pmax) continue;  // rows are not always ascending (nearest first)
        if (R >= 0 && cells_single_root(a.rcells[r], cmin, cmax, R)) continue;
        visit_range<T, D>(a.soa, a.ld, core, rsnap, qb, uniform(min(rg.y, pmax)), body, never);
    }
}

template <typename T, int D>
__global__ __launch_bounds__(kThreads) void k_border(const DbscanArgs<T> a,
                                                     const uint8_t* __restrict__ core,
                                                     const int32_t* __restrict__ root,
                                                     const int32_t* __restrict__ cmin,
                                                     const int32_t* __restrict__ cmax,
                                                     const uint32_t* __restrict__ order,
                                                     int64_t* __restrict__ labels,
                                                     unsigned long long* __restrict__ stats,
                                                     int2* __restrict__ amb_list) {
    Chunk c;
    if (!fetch_chunk(a.items, a.nitems, a.ustart, a.roff, c)) return;
    const JobParams<T>& jp = a.jobs[uniform(a.job_of_cell[c.u])];
    const T eps2 = jp.eps2;
    const int64_t first_pos = jp.row_begin;  // cluster ids are positions inside the job
    const int32_t p = c.first + lane_id();
    const bool valid = p < c.end;
    const bool active = valid && !core[p];
    if (!__any(active)) return;
    // do the candidate cells hold cores of a single root only?
    int32_t R = -1;
    bool single = true;
    for (int32_t r = c.r0; r < c.r1 && single; ++r) {
        const int2 cs = a.rcells[r];
        for (int32_t cc = cs.x; cc < cs.y; ++cc) {
            const int32_t mn = cmin[cc], mx = cmax[cc];
            if (mn > mx) continue;
            if (mn != mx || (R >= 0 && R != mn)) {
                single = false;
                break;
            }
            R = mn;
        }
    }
    R = uniform(R);
    int32_t best = INT_MAX, worst = -1;
    if (!(single && R < 0)) {  // otherwise no core is near: all noise
        T pc[D];
        load_row<T, D>(a.soa, a.ld, valid ? p : c.first, pc);
        auto body = [&](int32_t, const T* qc, uint8_t cq, int32_t rq) {
            if (!cq) return;
            if (active && within<D>(pc, qc, eps2)) {
                best = min(best, rq);
                worst = max(worst, rq);
            }
        };
        auto stop = [&] {
            return single && static_cast<bool>(__all(!active || best != INT_MAX));
        };
        const int32_t center = uniform(a.rcenter[c.u]);
        for (int32_t i = -1; i < c.r1 - c.r0; ++i) {
            const int32_t r = i < 0 ? center : c.r0 + i;
            if (i >= 0 && r == center) continue;
            const int2 rg = a.ranges[r];
            if (visit_range<T, D>(a.soa, a.ld, core, root, uniform(rg.x), uniform(rg.y), body,
                                  stop))
                break;
        }
    }
    if (active) labels[order[p]] = best == INT_MAX ? 0 : static_cast<int64_t>(best) - first_pos + 1;
    const bool is_amb = active && best != INT_MAX && best != worst;
    const uint64_t amb_mask = ballot(is_amb);
    const unsigned long long amb = __popcll(amb_mask);
    unsigned long long base = 0;
    if (lane_id() == 0) {
        if (amb) base = atomicAdd(&stats[1], amb);
    }
    // record (slot, cell) of every border row next to two or more clusters
    if (amb_list && amb) {
        base = __shfl(base, 0, 64);
        if (is_amb)
            amb_list[base + static_cast<unsigned long long>(__popcll(amb_mask & lanemask_lt()))] =
                make_int2(p, c.u);
    }
}

// Label of a non-core row (lanes where `on`) next to clusters from `best` to
// `worst` (INT_MAX and -1: none): the smallest, or noise (returns 1).  Rows next
// to two or more are counted in stats[1] and listed.  The whole wave calls it.
__device__ __forceinline__ unsigned int border_label(bool on, int32_t p, int32_t u,
                                                     const uint32_t* __restrict__ inrow,
                                                     int32_t best, int32_t worst, int64_t first_pos,
                                                     int64_t* __restrict__ labels,
                                                     unsigned long long* __restrict__ stats,
                                                     int2* __restrict__ amb_list) {
    if (on) labels[inrow[p]] = best == INT_MAX ? 0 : static_cast<int64_t>(best) - first_pos + 1;
    const bool is_amb = on && best != INT_MAX && best != worst;
    const uint64_t amb = ballot(is_amb);
    if (amb != 0) {
        unsigned long long at = 0;
        if (lane_id() == 0)
            at = atomicAdd(&stats[1], static_cast<unsigned long long>(__popcll(amb)));
        if (amb_list) {
            at = bcast64(at, 0);
            if (is_amb)
                amb_list[at + static_cast<unsigned long long>(__popcll(amb & lanemask_lt()))] =
                    make_int2(p, u);
        }
    }
    return on && best == INT_MAX ? 1u : 0u;
}

// Box-mode border labels: every core of a box lies in the box's cluster
// (bcluster), so a non-core row only needs, per neighbour box whose cluster
// could change its answer, one within-eps core of that box (or a box within
// eps as a whole).  G lanes per listed row, a box per lane, as in
// k_core_rows; a box is skipped when its cluster is the row's current one, or
// larger once two clusters were met; the smallest adjacent cluster and the
// two-cluster flag come out exact.  stats[0] += noise rows, stats[1] += rows
// next to two or more clusters.  Walks of boxes of more than kHeavyWalk rows
// are put off as in k_core_rows: the row's clusters so far go to a.slot_a and
// a.slot_b, k_border_heavy adds the parts' and k_border_late labels the row.
// Lanes per row (ms by lanes: 5M rows of 4 (16) 0.256, (32) 0.241, (64) 0.302;
// 30k of 6 doubles (16) 0.079, (32) 0.053, (64) 0.040).
// Float rows up to 3-D run at 7 waves per SIMD (4096 clouds of 8k rows: 6 waves
// 2.38 ms, 7 2.16, 8 2.24; 10M rows 101 us, 98, 114).
template <int D>
constexpr int kBorderGroup = D <= 3 ? 8 : D == 4 ? 32 : 64;
template <typename T, int D, bool kHeavy>
__global__ __launch_bounds__(kThreads, D <= 3 && sizeof(T) == 4 && !kHeavy ? 7 : 1)
void k_border_rows(
    const DbscanArgs<T> a, const uint8_t* __restrict__ core, const int32_t* __restrict__ bcluster,
    const int2* __restrict__ rows, const unsigned int* __restrict__ nrows_dev,
    int64_t* __restrict__ labels, unsigned long long* __restrict__ stats,
    int2* __restrict__ amb_list) {
    constexpr int G = kBorderGroup<D>;
    constexpr int kPer = 64 / G;
    const int32_t nrows = uniform(static_cast<int32_t>(*nrows_dev));
    const int gl = lane_id() & (G - 1);
    const Span<T>* bbox = static_cast<const Span<T>*>(a.bbox);
    unsigned long long noise = 0;
    for (int32_t base = first_wave() * kPer; base < nrows; base += wave_stride() * kPer) {
        const int32_t i = base + lane_id() / G;
        const bool on = i < nrows;
        const int2 it = rows[on ? i : nrows - 1];
        const int32_t p = it.x, u = it.y;
        T pc[D];
        load_row<T, D>(a.soa, a.ld, p, pc);
        const int32_t r0 = static_cast<int32_t>(a.roff[u]);
        const int32_t r1 = static_cast<int32_t>(a.roff[u + 1]);
        const JobParams<T>& jp = a.jobs[a.njobs == 1 ? 0 : a.job_of_cell[u]];
        const T eps2 = jp.eps2;
        int32_t best = INT_MAX, worst = -1;  // smallest, largest adjacent cluster so far
        bool put_off = false;                // the row has entries in a.heavy
        group_boxes<G>(on, r0, r1, a.rcenter[u], a.cbox[u], a.rboxes, 0, INT_MAX,
                       [&](bool valid, int32_t b) {
            const int32_t cl = valid ? bcluster[b] : -1;
            auto wanted = [&] { return cl >= 0 && cl != best && (cl < best || best == worst); };
            int32_t q0 = 0, q1 = 0;
            bool part = false, hit = false;
            if (wanted()) {
                T gmin2, gmax2;
                point_box<T, D>(bbox, b, pc, gmin2, gmax2);
                q0 = a.bstart[b];
                q1 = a.bstart[b + 1];
                const bool near = gmin2 <= eps2;
                hit = near && gmax2 <= eps2;
                part = near && !hit;
            }
            if (__any(hit)) {
                best = min(best, group_min<G>(hit ? cl : INT_MAX));
                worst = max(worst, group_max<G>(hit ? cl : -1));
            }
            const bool lane_walk = q1 - q0 <= kLaneRows;
            if (__any(part)) {
                bool h = false;
                if (part && lane_walk && wanted()) {
                    for (int32_t q = q0; q < q1 && !h; ++q) {
                        if (!core[q]) continue;
                        T qc[D];
                        load_row<T, D>(a.soa, a.ld, q, qc);
                        h = within<D>(pc, qc, eps2);
                    }
                }
                if (__any(h)) {
                    best = min(best, group_min<G>(h ? cl : INT_MAX));
                    worst = max(worst, group_max<G>(h ? cl : -1));
                }
                for (uint64_t todo = ballot(part && !lane_walk && wanted()); todo != 0;
                     todo &= todo - 1) {
                    const int j = static_cast<int>(__builtin_ctzll(todo));
                    if (!((ballot(wanted()) >> j) & 1)) continue;
                    const int32_t v0 = bcast(q0, j), v1 = bcast(q1, j);
                    if constexpr (kHeavy)
                        if (v1 - v0 > kHeavyWalk && put_heavy(a, bcast(p, j), v0, v1)) {
                            if (lane_id() / G == j / G) put_off = true;
                            continue;
                        }
                    T pr[D];
#pragma unroll
                    for (int e = 0; e < D; ++e) pr[e] = bcast(pc[e], j);
                    uint32_t visited = 0;
                    if (wide_count<T, D>(a.soa, a.ld, core, v0, v1, pr, bcast(eps2, j), 1u,
                                         visited) != 0) {
                        const int32_t c = bcast(cl, j);
                        if (lane_id() / G == j / G) {
                            best = min(best, c);
                            worst = max(worst, c);
                        }
                    }
                }
            }
            return false;
        });
        if constexpr (kHeavy)
            if (on && gl == 0 && put_off) {
                a.slot_a[p] = best;
                a.slot_b[p] = worst;
                a.late[atomicAdd(a.nlate, 1u)] = p;
            }
        noise += border_label(on && gl == 0 && !put_off, p, u, a.inrow, best, worst, jp.row_begin,
                              labels, stats, amb_list);
    }
    block_add<kThreads>(noise, &stats[0]);
}

// The put-off walks of k_border_rows, a wave per entry.
template <typename T, int D>
__global__ __launch_bounds__(kThreads) void k_border_heavy(const DbscanArgs<T> a,
                                                           const uint8_t* __restrict__ core,
                                                           const int32_t* __restrict__ bcluster) {
    const int32_t n = heavy_count(a);
    for (int32_t w = first_wave(); w < n; w += wave_stride()) {
        const int32_t p = uniform(a.heavy[w].x), q0 = uniform(a.heavy[w].y);
        if (p < 0) continue;
        const int32_t b2 = uniform(a.box_of_slot[q0]);
        const int32_t cl = uniform(bcluster[b2]);
        const int32_t best = uniform(ld_agent(&a.slot_a[p]));
        const int32_t worst = uniform(ld_agent(&a.slot_b[p]));
        if (cluster_settled(best, worst, cl)) continue;
        const int32_t q1 = min(q0 + kHeavyWalk, uniform(a.bstart[b2 + 1]));
        const T eps2 = a.jobs[uniform(a.job_of_cell[uniform(a.bcell[b2])])].eps2;
        T pc[D];
        load_row<T, D>(a.soa, a.ld, p, pc);
        uint32_t visited = 0;
        if (wide_count<T, D>(a.soa, a.ld, core, q0, q1, pc, eps2, 1u, visited) == 0) continue;
        if (lane_id() == 0) {
            atomicMin(&a.slot_a[p], cl);
            atomicMax(&a.slot_b[p], cl);
        }
    }
}

template <typename T>
__global__ __launch_bounds__(kThreads) void k_border_late(const DbscanArgs<T> a,
                                                          int64_t* __restrict__ labels,
                                                          unsigned long long* __restrict__ stats,
                                                          int2* __restrict__ amb_list) {
    const int32_t n = static_cast<int32_t>(*a.nlate);
    unsigned long long noise = 0;
    const int32_t stride = static_cast<int32_t>(gridDim.x) * kThreads;
    for (int32_t i0 = static_cast<int32_t>(blockIdx.x) * kThreads; i0 < n; i0 += stride) {
        const int32_t i = i0 + static_cast<int32_t>(threadIdx.x);
        const bool on = i < n;
        const int32_t p = a.late[on ? i : 0];
        const int32_t u = a.bcell[a.box_of_slot[p]];
        noise += border_label(on, p, u, a.inrow, a.slot_a[p], a.slot_b[p],
                              a.jobs[a.job_of_cell[u]].row_begin, labels, stats, amb_list);
    }
    block_add<kThreads>(noise, &stats[0]);
}

// ---------------------------------------------------------------------------
// The reference's border choice at one thread (HPD_BORDER_ONE_THREAD).
//
// Processing rows in sorted order, the reference gives core c the
// provisional label f(c) + 1 with f(c) = min(pos(c), f(q) over within-eps
// cores q before c) (hpdbscan.h:74-92 with spatial_index.h:757-763), i.e. the
// smallest position reachable from c along strictly decreasing positions.
// A border row keeps the smallest provisional label among its adjacent cores
// (the atomic_min of hpdbscan.h:91) and ends in that core's cluster.  Only
// border rows next to two or more clusters depend on it; f is computed for
// the cores of the clusters they touch, by in-place relaxation to the fixed
// point.
// ---------------------------------------------------------------------------

// clusters touched by the ambiguous border rows -> involved[cluster] = 1
template <typename T, int D>
__global__ __launch_bounds__(kThreads) void k_ot_mark(const DbscanArgs<T> a,
                                                      const uint8_t* __restrict__ core,
                                                      const int32_t* __restrict__ rootslot,
                                                      const int2* __restrict__ amb, int32_t namb,
                                                      uint8_t* __restrict__ involved) {
    const int32_t i = static_cast<int32_t>(blockIdx.x) * kThreads + threadIdx.x;
    if (i >= namb) return;
    const int32_t p = amb[i].x, u = amb[i].y;
    const T eps2 = a.jobs[a.job_of_cell[u]].eps2;
    T pc[D];
    load_row<T, D>(a.soa, a.ld, p, pc);
    for (uint32_t r = a.roff[u]; r < a.roff[u + 1]; ++r) {
        const int2 rg = a.ranges[r];
        for (int32_t q = rg.x; q < rg.y; ++q) {
            if (!core[q]) continue;
            T qc[D];
            load_row<T, D>(a.soa, a.ld, q, qc);
            if (within<D>(pc, qc, eps2)) involved[rootslot[q]] = 1;
        }
    }
}

// one in-place relaxation sweep of f over the cores of involved clusters;
// f is indexed by slot and holds positions
template <typename T, int D>
__global__ __launch_bounds__(kThreads) void k_ot_relax(const DbscanArgs<T> a,
                                                       const uint8_t* __restrict__ core,
                                                       const int32_t* __restrict__ rootslot,
                                                       const uint8_t* __restrict__ involved,
                                                       int32_t* f, unsigned int* __restrict__ changed) {
    Chunk c;
    if (!fetch_chunk(a.items, a.nitems, a.ustart, a.roff, c)) return;
    const int32_t p = c.first + lane_id();
    const bool valid = p < c.end;
    const bool active = valid && core[p] && involved[rootslot[p]];
    if (!__any(active)) return;
    const T eps2 = a.jobs[uniform(a.job_of_cell[c.u])].eps2;
    const int32_t pp = valid ? slot_pos(a.pos_of_slot, p) : 0;
    T pc[D];
    load_row<T, D>(a.soa, a.ld, valid ? p : c.first, pc);
    int32_t fmin = active ? ld_agent(&f[p]) : INT_MAX;
    const int32_t f0 = fmin;
    for (int32_t r = c.r0; r < c.r1; ++r) {
        const int2 rg = a.ranges[r];
        const int32_t qb = uniform(rg.x), qe = uniform(rg.y);
        // a row starting past the chunk's cell holds later positions only;
        // rows are not always ascending (nearest first), so skip, not stop
        if (qb >= c.end) continue;
        for (int32_t q = qb; q < qe; ++q) {
            if (!core[q]) continue;
            const int32_t qp = slot_pos(a.pos_of_slot, q);
            T qc[D];
            load_row<T, D>(a.soa, a.ld, q, qc);
            if (active && qp < pp && within<D>(pc, qc, eps2)) fmin = min(fmin, ld_agent(&f[q]));
        }
    }
    if (active && fmin < f0) {
        st_agent(&f[p], fmin);
        atomicOr(changed, 1u);
    }
}

// final choice for every ambiguous border row: the cluster of the adjacent
// core with the smallest f
template <typename T, int D>
__global__ __launch_bounds__(kThreads) void k_ot_assign(const DbscanArgs<T> a,
                                                        const uint8_t* __restrict__ core,
                                                        const int32_t* __restrict__ rootslot,
                                                        const int2* __restrict__ amb, int32_t namb,
                                                        const int32_t* __restrict__ f,
                                                        int64_t* __restrict__ labels) {
    const int32_t i = static_cast<int32_t>(blockIdx.x) * kThreads + threadIdx.x;
    if (i >= namb) return;
    const int32_t p = amb[i].x, u = amb[i].y;
    const JobParams<T>& jp = a.jobs[a.job_of_cell[u]];
    T pc[D];
    load_row<T, D>(a.soa, a.ld, p, pc);
    int32_t best_f = INT_MAX, best_cluster = -1;
    for (uint32_t r = a.roff[u]; r < a.roff[u + 1]; ++r) {
        const int2 rg = a.ranges[r];
        for (int32_t q = rg.x; q < rg.y; ++q) {
            if (!core[q]) continue;
            T qc[D];
            load_row<T, D>(a.soa, a.ld, q, qc);
            if (within<D>(pc, qc, jp.eps2) && f[q] < best_f) {
                best_f = f[q];
                best_cluster = rootslot[q];
            }
        }
    }
    if (best_cluster >= 0)
        labels[a.inrow[p]] = static_cast<int64_t>(best_cluster) - jp.row_begin + 1;
}

__global__ __launch_bounds__(kThreads) void k_ot_init(const uint8_t* __restrict__ core,
                                                      const uint32_t* __restrict__ pos_of_slot,
                                                      int32_t* __restrict__ f, int64_t n) {
    const int64_t i = static_cast<int64_t>(blockIdx.x) * kThreads + threadIdx.x;
    if (i < n) f[i] = core[i] ? slot_pos(pos_of_slot, static_cast<int32_t>(i)) : INT_MAX;
}

// Number of zero labels among labels[0, n): one atomic per block.
__global__ __launch_bounds__(kThreads) void k_count_zero(const int64_t* __restrict__ v, int64_t n,
                                                         unsigned long long* __restrict__ out) {
    __shared__ unsigned long long part[kWavesPerBlock];
    unsigned long long c = 0;
    for (int64_t i = static_cast<int64_t>(blockIdx.x) * kThreads + threadIdx.x; i < n;
         i += static_cast<int64_t>(gridDim.x) * kThreads)
        c += v[i] == 0 ? 1ull : 0ull;
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) c += __shfl_xor(c, o, 64);
    if (lane_id() == 0) part[threadIdx.x >> 6] = c;
    __syncthreads();
    if (threadIdx.x == 0) {
        unsigned long long t = 0;
#pragma unroll
        for (int w = 0; w < kWavesPerBlock; ++w) t += part[w];
        if (t) atomicAdd(out, t);
    }
}

// Sum of n byte flags (0/1): one atomic per block.
__global__ __launch_bounds__(kThreads) void k_count_flags(const uint8_t* __restrict__ f, int64_t n,
                                                          unsigned long long* __restrict__ out) {
    __shared__ unsigned long long part[kWavesPerBlock];
    unsigned long long c = 0;
    for (int64_t i = static_cast<int64_t>(blockIdx.x) * kThreads + threadIdx.x; i < n;
         i += static_cast<int64_t>(gridDim.x) * kThreads)
        c += f[i];
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) c += __shfl_xor(c, o, 64);
    if (lane_id() == 0) part[threadIdx.x >> 6] = c;
    __syncthreads();
    if (threadIdx.x == 0) {
        unsigned long long t = 0;
#pragma unroll
        for (int w = 0; w < kWavesPerBlock; ++w) t += part[w];
        if (t) atomicAdd(out, t);
    }
}

__global__ __launch_bounds__(kThreads) void k_iota(int32_t* __restrict__ v, int64_t n) {
    const int64_t i = static_cast<int64_t>(blockIdx.x) * kThreads + threadIdx.x;
    if (i < n) v[i] = static_cast<int32_t>(i);
}

__global__ __launch_bounds__(kThreads) void k_fill2(int32_t* __restrict__ a, int32_t va,
                                                    int32_t* __restrict__ b, int32_t vb, int64_t n) {
    const int64_t i = static_cast<int64_t>(blockIdx.x) * kThreads + threadIdx.x;
    if (i < n) {
        a[i] = va;
        b[i] = vb;
    }
}

inline unsigned blocks_for(int64_t n, int t) { return static_cast<unsigned>((n + t - 1) / t); }

}  // namespace

// *out += number of nonzero flags among f[0, n)
static void count_flags(const uint8_t* f, int64_t n, unsigned long long* out, hipStream_t s) {
    if (n <= 0) return;
    const int64_t want = (n + kThreads - 1) / kThreads;
    const unsigned grid = static_cast<unsigned>(want < 2048 ? want : 2048);
    hipLaunchKernelGGL(k_count_flags, dim3(grid), dim3(kThreads), 0, s, f, n, out);
    HPD_HIP(hipGetLastError());
}

// *out += number of zero labels (noise rows) among labels[0, n)
static void count_noise(const int64_t* labels, int64_t n, unsigned long long* out, hipStream_t s) {
    if (n <= 0) return;
    const int64_t want = (n + kThreads - 1) / kThreads;
    const unsigned grid = static_cast<unsigned>(want < 2048 ? want : 2048);
    hipLaunchKernelGGL(k_count_zero, dim3(grid), dim3(kThreads), 0, s, labels, n, out);
    HPD_HIP(hipGetLastError());
}

#if !defined(HPD_DBSCAN_PART) || HPD_DBSCAN_PART == 0
int32_t heavy_walk_rows() { return kHeavyWalk; }
#endif

template <typename T, int D>
void launch_core(const DbscanArgs<T>& a, uint8_t* core, unsigned long long* ntests, hipStream_t s,
                 hipEvent_t count_start) {
    unsigned long long* ncore = nullptr;  // (the other core kernels count nothing)
    if (count_start) HPD_HIP(hipEventRecord(count_start, s));  // (no box pass: all of it)
    if constexpr (std::is_floating_point<T>::value) {
        if (a.bbox) {
            // rows of tight boxes with >= minPts rows are core, every other
            // row starts non-core; the rows that can be core are listed
            launch_core_init(a.n, a.box_of_slot, a.btight, a.bstart, a.bcell, a.inrow, core,
                             a.bmincore, a.crows, a.ncrows_dev, kGroup<D>, s);
            if (count_start) HPD_HIP(hipEventRecord(count_start, s));
            constexpr int per_wave = 64 / kGroup<D>;
            auto rows = [&](auto count, auto heavy) {
                constexpr auto kernel = k_core_rows<T, D, decltype(count)::value,
                                                    decltype(heavy)::value>;
                hipLaunchKernelGGL(kernel, dim3(persistent_blocks<kernel>(a.n, per_wave)),
                                   dim3(kThreads), 0, s, a, core, ntests);
            };
            if (ntests) rows(std::true_type{}, std::true_type{});
            else if (a.heavy_cap > 0) rows(std::false_type{}, std::true_type{});
            else rows(std::false_type{}, std::false_type{});
            if (a.heavy_cap > 0)
                hipLaunchKernelGGL((k_core_heavy<T, D>),
                                   dim3(persistent_blocks<k_core_heavy<T, D>>(a.n, 1)),
                                   dim3(kThreads), 0, s, a, core, ntests);
            HPD_HIP(hipGetLastError());
            return;
        }
    }
    if (a.nitems <= 0) return;
    hipLaunchKernelGGL((k_core<T, D>), dim3(blocks_for(a.nitems, kWavesPerBlock)), dim3(kThreads),
                       0, s, a, core, ncore);
    HPD_HIP(hipGetLastError());
}

template <typename T, int D, typename K>
void launch_label_full_rows(const T* pts, const DbscanArgs<T>& a, int sub_k, int sub_bits,
                            const K* keys, Count nbox, const int32_t* bcluster, int32_t* tab,
                            int64_t cap, int64_t* labels, unsigned int* ok, hipStream_t s) {
    if (a.n <= 0 || nbox.host <= 0) return;
    hipLaunchKernelGGL((k_full_box_table<T, K>), dim3(blocks_for(nbox.host, kThreads)),
                       dim3(kThreads), 0, s, keys, a.n, a.bstart, nbox, a.bcell, a.job_of_cell,
                       a.jobs, a.btight, bcluster, tab, cap, ok);
    hipLaunchKernelGGL((k_label_full_rows<T, D, K>),
                       dim3(blocks_for(a.n, kWavesPerBlock * kFullRows)),
                       dim3(kThreads), 0, s, pts, a.n,
                       a.jobs, a.njobs, sub_k, sub_bits, static_cast<const int32_t*>(tab), cap,
                       static_cast<const unsigned int*>(ok), labels);
    HPD_HIP(hipGetLastError());
}

template <typename T, int D>
void launch_union_points(const DbscanArgs<T>& a, const uint8_t* core, int32_t* parent,
                         int32_t* rsnap, int32_t* cmin, int32_t* cmax, int32_t* compmin,
                         hipStream_t s) {
    if (a.n <= 0) return;
    const unsigned gw = blocks_for(a.nitems, kWavesPerBlock);
    hipLaunchKernelGGL(k_iota, dim3(blocks_for(a.n, kThreads)), dim3(kThreads), 0, s, parent, a.n);
    hipLaunchKernelGGL((k_hook<T, D>), dim3(gw), dim3(kThreads), 0, s, a, core, parent);
    hipLaunchKernelGGL(k_fill2, dim3(blocks_for(a.m, kThreads)), dim3(kThreads), 0, s, cmin, INT_MAX,
                       cmax, -1, static_cast<int64_t>(a.m));
    hipLaunchKernelGGL(k_roots, dim3(gw), dim3(kThreads), 0, s, a.items, a.nitems, a.ustart, a.roff,
                       core, parent, rsnap, cmin, cmax);
    hipLaunchKernelGGL((k_union<T, D>), dim3(gw), dim3(kThreads), 0, s, a, core,
                       static_cast<const int32_t*>(rsnap), static_cast<const int32_t*>(cmin),
                       static_cast<const int32_t*>(cmax), parent);
    hipLaunchKernelGGL(k_fill2, dim3(blocks_for(a.n, kThreads)), dim3(kThreads), 0, s, compmin,
                       INT_MAX, rsnap, 0, a.n);
    hipLaunchKernelGGL(k_compmin, dim3(blocks_for(a.n, kThreads)), dim3(kThreads), 0, s, core,
                       parent, a.n, a.pos_of_slot, compmin);
    HPD_HIP(hipGetLastError());
}

template <typename T>
void launch_label_cores(const DbscanArgs<T>& a, const uint8_t* core, const int32_t* bcluster,
                        int32_t* parent, const int32_t* compmin, int32_t* rootslot, int32_t* cmin,
                        int32_t* cmax, int64_t* labels, unsigned long long* ncore, hipStream_t s,
                        const unsigned int* full_ok) {
    if (a.n <= 0) return;
    if (bcluster && a.bcell) {
        hipLaunchKernelGGL(k_label_cores_boxes<T>, dim3(collect_blocks(a.n)), dim3(kThreads), 0, s,
                           a.n, a.jobs, a.job_of_cell, core, a.box_of_slot, a.bcell, bcluster,
                           a.inrow, labels, rootslot, ncore, a.njobs == 1,
                           full_ok ? a.btight : nullptr, full_ok, a.brows, a.nbrows_dev);
        HPD_HIP(hipGetLastError());
        return;
    }
    const unsigned gw = blocks_for(a.nitems, kWavesPerBlock);
    count_flags(core, a.n, ncore, s);
    hipLaunchKernelGGL(k_fill2, dim3(blocks_for(a.m, kThreads)), dim3(kThreads), 0, s, cmin, INT_MAX,
                       cmax, -1, static_cast<int64_t>(a.m));
    hipLaunchKernelGGL(k_label_cores<T>, dim3(gw), dim3(kThreads), 0, s, a.items, a.nitems,
                       a.ustart, a.roff, a.jobs, a.job_of_cell, core, a.box_of_slot, bcluster,
                       parent, compmin, a.inrow, labels, rootslot, cmin, cmax);
    HPD_HIP(hipGetLastError());
}

template <typename T, int D>
void launch_border(const DbscanArgs<T>& a, const uint8_t* core, const int32_t* bcluster,
                   const int32_t* rootslot, const int32_t* cmin, const int32_t* cmax,
                   int64_t* labels, unsigned long long* stats, int2* amb_list, hipStream_t s) {
    if (a.n <= 0) return;
    const unsigned gw = blocks_for(a.nitems, kWavesPerBlock);
    if constexpr (std::is_floating_point<T>::value) {
        if (bcluster && a.bbox) {
            auto rows = [&](auto heavy) {
                constexpr auto kernel = k_border_rows<T, D, decltype(heavy)::value>;
                hipLaunchKernelGGL(kernel, dim3(persistent_blocks<kernel>(a.n, 64 / kBorderGroup<D>)),
                                   dim3(kThreads), 0, s, a, core, bcluster,
                                   static_cast<const int2*>(a.brows),
                                   static_cast<const unsigned int*>(a.nbrows_dev), labels, stats,
                                   amb_list);
            };
            if (a.heavy_cap > 0) rows(std::true_type{});
            else rows(std::false_type{});
            if (a.heavy_cap > 0) {
                hipLaunchKernelGGL((k_border_heavy<T, D>),
                                   dim3(persistent_blocks<k_border_heavy<T, D>>(a.n, 1)),
                                   dim3(kThreads), 0, s, a, core, bcluster);
                hipLaunchKernelGGL(k_border_late<T>, dim3(256), dim3(kThreads), 0, s, a, labels,
                                   stats, amb_list);
            }
            HPD_HIP(hipGetLastError());
            return;
        }
    }
    hipLaunchKernelGGL((k_border<T, D>), dim3(gw), dim3(kThreads), 0, s, a, core, rootslot, cmin,
                       cmax, a.inrow, labels, stats, amb_list);
    HPD_HIP(hipGetLastError());
    count_noise(labels, a.n, &stats[0], s);
}

template <typename T, int D>
void launch_one_thread_mark(const DbscanArgs<T>& a, const uint8_t* core, const int32_t* rootslot,
                            const int2* amb, int32_t namb, uint8_t* involved, int32_t* f,
                            hipStream_t s) {
    hipLaunchKernelGGL((k_ot_mark<T, D>), dim3(blocks_for(namb, kThreads)), dim3(kThreads), 0, s,
                       a, core, rootslot, amb, namb, involved);
    hipLaunchKernelGGL(k_ot_init, dim3(blocks_for(a.n, kThreads)), dim3(kThreads), 0, s, core,
                       a.pos_of_slot, f, a.n);
    HPD_HIP(hipGetLastError());
}

template <typename T, int D>
void launch_one_thread_relax(const DbscanArgs<T>& a, const uint8_t* core, const int32_t* rootslot,
                             const uint8_t* involved, int32_t* f, unsigned int* changed,
                             hipStream_t s) {
    hipLaunchKernelGGL((k_ot_relax<T, D>), dim3(blocks_for(a.nitems, kWavesPerBlock)),
                       dim3(kThreads), 0, s, a, core, rootslot, involved, f, changed);
    HPD_HIP(hipGetLastError());
}

template <typename T, int D>
void launch_one_thread_assign(const DbscanArgs<T>& a, const uint8_t* core, const int32_t* rootslot,
                              const int2* amb, int32_t namb, const int32_t* f, int64_t* labels,
                              hipStream_t s) {
    hipLaunchKernelGGL((k_ot_assign<T, D>), dim3(blocks_for(namb, kThreads)), dim3(kThreads), 0, s,
                       a, core, rootslot, amb, namb, f, labels);
    HPD_HIP(hipGetLastError());
}

#define HPD_INST_DBSCAN(T, D)                                                                     \
    template void launch_core<T, D>(const DbscanArgs<T>&, uint8_t*, unsigned long long*,          \
                                    hipStream_t, hipEvent_t);                                     \
    template void launch_union_points<T, D>(const DbscanArgs<T>&, const uint8_t*, int32_t*,       \
                                            int32_t*, int32_t*, int32_t*, int32_t*, hipStream_t); \
    template void launch_border<T, D>(const DbscanArgs<T>&, const uint8_t*, const int32_t*,       \
                                      const int32_t*, const int32_t*, const int32_t*, int64_t*,   \
                                      unsigned long long*, int2*, hipStream_t);                   \
    template void launch_one_thread_mark<T, D>(const DbscanArgs<T>&, const uint8_t*,              \
                                               const int32_t*, const int2*, int32_t, uint8_t*,    \
                                               int32_t*, hipStream_t);                            \
    template void launch_one_thread_relax<T, D>(const DbscanArgs<T>&, const uint8_t*,             \
                                                const int32_t*, const uint8_t*, int32_t*,         \
                                                unsigned int*, hipStream_t);                      \
    template void launch_one_thread_assign<T, D>(const DbscanArgs<T>&, const uint8_t*,            \
                                                 const int32_t*, const int2*, int32_t,            \
                                                 const int32_t*, int64_t*, hipStream_t);
#define HPD_INST_DBSCAN_ALL_D(T) \
    HPD_INST_DBSCAN(T, 1)        \
    HPD_INST_DBSCAN(T, 2)        \
    HPD_INST_DBSCAN(T, 3)        \
    HPD_INST_DBSCAN(T, 4)        \
    HPD_INST_DBSCAN(T, 5)        \
    HPD_INST_DBSCAN(T, 6)        \
    HPD_INST_DBSCAN(T, 7)        \
    HPD_INST_DBSCAN(T, 8)

// The build compiles this file in parts (HPD_DBSCAN_PART), each a share of
// the element types, so that they compile in parallel.
#ifndef HPD_DBSCAN_PART
#define HPD_DBSCAN_PART 0
#endif
#if HPD_DBSCAN_PART == 0
#define HPD_FOR_EACH_PART_DTYPE(X) X(float)
#elif HPD_DBSCAN_PART == 1
#define HPD_FOR_EACH_PART_DTYPE(X) X(double)
#elif HPD_DBSCAN_PART == 2
#define HPD_FOR_EACH_PART_DTYPE(X) X(int8_t) X(int16_t) X(int32_t) X(int64_t)
#else
#define HPD_FOR_EACH_PART_DTYPE(X) X(uint8_t) X(uint16_t) X(uint32_t) X(uint64_t)
#endif

HPD_FOR_EACH_PART_DTYPE(HPD_INST_DBSCAN_ALL_D)

#define HPD_INST_LABEL_CORES(T)                                                                \
    template void launch_label_cores<T>(const DbscanArgs<T>&, const uint8_t*, const int32_t*,  \
                                        int32_t*, const int32_t*, int32_t*, int32_t*, int32_t*, \
                                        int64_t*, unsigned long long*, hipStream_t,      \
                                        const unsigned int*);
HPD_FOR_EACH_PART_DTYPE(HPD_INST_LABEL_CORES)

#define HPD_INST_FULL_ROWS(T, D, K)                                                             \
    template void launch_label_full_rows<T, D, K>(const T*, const DbscanArgs<T>&, int, int,     \
                                                  const K*, Count, const int32_t*, int32_t*,     \
                                                  int64_t, int64_t*, unsigned int*, hipStream_t);
#define HPD_INST_FULL_ROWS_ALL(T)          \
    HPD_INST_FULL_ROWS(T, 1, uint32_t)     \
    HPD_INST_FULL_ROWS(T, 2, uint32_t)     \
    HPD_INST_FULL_ROWS(T, 3, uint32_t)     \
    HPD_INST_FULL_ROWS(T, 4, uint32_t)     \
    HPD_INST_FULL_ROWS(T, 5, uint32_t)     \
    HPD_INST_FULL_ROWS(T, 6, uint32_t)     \
    HPD_INST_FULL_ROWS(T, 7, uint32_t)     \
    HPD_INST_FULL_ROWS(T, 8, uint32_t)     \
    HPD_INST_FULL_ROWS(T, 1, uint64_t)     \
    HPD_INST_FULL_ROWS(T, 2, uint64_t)     \
    HPD_INST_FULL_ROWS(T, 3, uint64_t)     \
    HPD_INST_FULL_ROWS(T, 4, uint64_t)     \
    HPD_INST_FULL_ROWS(T, 5, uint64_t)     \
    HPD_INST_FULL_ROWS(T, 6, uint64_t)     \
    HPD_INST_FULL_ROWS(T, 7, uint64_t)     \
    HPD_INST_FULL_ROWS(T, 8, uint64_t)
#if HPD_DBSCAN_PART == 0
HPD_INST_FULL_ROWS_ALL(float)
#elif HPD_DBSCAN_PART == 1
HPD_INST_FULL_ROWS_ALL(double)
#endif


}  // namespace hpd
