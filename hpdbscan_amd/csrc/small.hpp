// Launcher of the kernels for small inputs (small.hip).
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

#include "internal.hpp"

namespace hpd {

// What a small run leaves behind.
struct SmallResult {
    unsigned long long sum_candidates;
    unsigned long long cores;
    unsigned long long noise;
    unsigned long long ambiguous;
    unsigned long long cells;         // occupied cells
    unsigned long long boxes;         // occupied sub-boxes
    unsigned long long neighbor_rows;
    unsigned long long total_cells;   // of the grid
    unsigned int nonfinite;           // a coordinate is NaN or infinite
    unsigned int overflow;            // the grid has more than 2^64 cells
    unsigned int unfit;               // a dimension of 2^31 cells or more
    unsigned int blocks_done;
};

// Most rows of a small run.  All pairs of rows are compared, so the time grows
// with their square; the general path costs some 35 launches whatever the
// size.
int64_t small_rows(int d);

template <typename T, int D>
size_t small_workspace_bytes(int64_t n);

// Labels of n <= small_rows(D) rows of one job (jp: eps2, min_pts and
// reciprocals; jp_dev, when not null, holds them in device memory instead)
// under the smallest-cluster border rule, by comparing all pairs: no sort, no
// index, no read-back.  work: small_workspace_bytes.  The result is
// gathered in *result (device memory) and written to *host (host memory mapped
// into the device) by the last kernel; with its nonfinite, overflow or unfit
// set the labels are not written.
template <typename T, int D>
void launch_small(const T* pts, int64_t n, const JobParams<T>& jp, const JobParams<T>* jp_dev,
                  int sub_k, int sub_bits, void* work, SmallResult* result, SmallResult* host,
                  int64_t* labels, hipStream_t s);

}  // namespace hpd
