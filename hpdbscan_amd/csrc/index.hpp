// Launchers of the occupied-cell and neighbour-range kernels (index.hip).
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

#include "internal.hpp"

namespace hpd {

// Cells of sorted keys whose cell id is key >> shift.  flags must hold
// 2*n + 1 uint32 (run flags, then their exclusive scan); writes ucell[0..m),
// ustart[0..m] with ustart[m] = n, and m to *ncells_dev.
template <typename K>
void launch_cells(const K* keys, int64_t n, int shift, uint32_t* flags, uint32_t* scan_tmp,
                  K* ucell, int32_t* ustart, uint32_t* ncells_dev, hipStream_t s);

// job_of_cell[u] = job of cell u; nranges[u] = number of non-empty
// neighbour rows of cell u; cell_core[u] (when not null) = 1 if cell u has
// >= minPts candidates (only then can it hold cores), else 0; adds
// Σ_u count(u) * |candidates(u)| to *sumcand and Σ_u nranges[u] to
// *rows_total (64-bit, unlike the scan of nranges).  max_rows = 3^(D-1), the
// most neighbour rows a cell can have.  With a stash (m * max_rows entries) the
// rows' cell ranges go to stash[u * max_rows ..] and the own row's index
// among them to rcenter[u], for launch_neighbor_copy; with by_class (D <= 4)
// each row's offset class (the number of dimensions it is offset in) rides
// in the top bits of its two cell indices.
template <typename K, typename T>
void launch_neighbor_count(const K* ucell, const int32_t* ustart, Count m,
                           const JobParams<T>* jobs, int32_t njobs, int32_t* job_of_cell,
                           uint32_t* nranges, uint8_t* cell_core, unsigned long long* sumcand,
                           unsigned long long* rows_total, int2* stash, int32_t max_rows,
                           int32_t* rcenter, bool by_class, hipStream_t s,
                           const int32_t* ctab = nullptr);

// Box mode: launch_neighbor_fill's box ranges and rcenter from the count
// pass's stash (roff scanned); with by_class the rows of each cell go
// nearest first (own row, then by the number of offset dimensions) instead of
// ascending
void launch_neighbor_copy(const int2* stash, int32_t stash_rows, int32_t m, const uint32_t* roff,
                          const int32_t* cbox, int2* rboxes, int32_t* rcenter, bool by_class,
                          hipStream_t s);

// ranges[roff[u] ..) = [first row, end row) of each non-empty neighbour row,
// ascending; rcells[..] = [first, end) occupied-cell index of the same row;
// rcenter[u] = index (into ranges) of the row holding cell u itself.  With
// cbox (first box of every cell) rcells gets the rows' box ranges
// [cbox[first], cbox[end]) instead: the box kernels then read them in one
// load, not three dependent ones.  ranges may be null.
template <typename K, typename T>
void launch_neighbor_fill(const K* ucell, const int32_t* ustart, Count m,
                          const JobParams<T>* jobs, int32_t* job_of_cell, uint32_t* roff,
                          int2* ranges, int2* rcells, int32_t* rcenter, int32_t max_rows,
                          hipStream_t s, const int32_t* ctab = nullptr,
                          const int32_t* cbox = nullptr);
// Whether the two take few cells by groups of lanes (no stash then: the fill
// searches again).
bool neighbor_rows_wide(int64_t cells, int32_t max_rows);

void launch_chunk_counts(const int32_t* ustart, Count m, uint32_t* nchunks, hipStream_t s);

// items[w] = (g, start[g] + 64 * (w - off[g])) for the `total` 64-row chunks
// of ngroups groups (off: exclusive scan of chunk counts, ngroups + 1 entries)
void launch_expand_chunks(const uint32_t* off, Count ngroups, const int32_t* start, Count total,
                          int2* items, hipStream_t s);
void launch_work_items(const int32_t* ustart, Count m, const uint32_t* coff, Count nitems,
                       int2* items, hipStream_t s);

}  // namespace hpd
