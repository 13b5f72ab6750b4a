// Launchers of the sub-box kernels (boxes.hip).
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

#include "internal.hpp"

namespace hpd {

// boxes per cell and dimension (k) and bits of the sub-box digit
int box_split(int d);
int box_sub_bits(int d);
int box_sub_bits(int d, int k);  // bits of the sub-box digit with k parts per dimension

template <typename T>
struct BoxArgs {
    const T* soa = nullptr;            // coordinates in slot order, [D][ld]
    int64_t ld = 0;
    int32_t nbox = 0;
    const uint32_t* nbox_dev = nullptr;  // static pipeline: nbox in device memory (nbox a bound)
    const int32_t* bstart = nullptr;   // first slot of every box, [nbox + 1]
    const int32_t* bcell = nullptr;    // occupied cell of every box
    const int32_t* cbox = nullptr;     // first box of every cell, [m + 1]
    void* bbox = nullptr;              // ordered-key min/max per box and dim
    const JobParams<T>* jobs = nullptr;
    int32_t njobs = 1;
    int64_t nrows = 0;
    const int32_t* job_of_cell = nullptr;
    const int32_t* rcenter = nullptr;  // index of every cell's own neighbour row
};

// coordinates in slot order (soa[j * ld + s] = pts[inrow_of_slot[s] * D + j];
// with pts null they are there already) and the bounding box of every box
// (bbox, 2 * D ordered keys per box, all written); part holds
// gather_part_bytes(n, D, sizeof(T)) bytes of scratch
template <typename T, int D>
void launch_gather_boxes(const T* pts, int64_t n, const uint32_t* inrow_of_slot, T* soa,
                         int64_t ld, const int32_t* box_of_slot, const int32_t* bstart, void* bbox,
                         void* part, hipStream_t s);
size_t gather_part_bytes(int64_t n, int d, int value_bytes);

// Boxes of keys sorted by (cell, sub-box digit) and the occupied cells: runs
// of equal keys, and of equal key >> shift (cell ids).  Writes the box of every
// slot; per box bstart (bstart[nbox] = n) and bcell; per cell ucell (its id),
// ustart (ustart[m] = n), cbox (first box; cbox[m] = nbox) and, with ctab,
// ctab[id]; *nbox_dev and *ncells_dev.  sums: scratch, max(2, n) words.
template <typename K>
void launch_box_table(const K* keys, int64_t n, int shift, uint32_t* sums, int32_t* box_of_slot,
                      int32_t* bstart, int32_t* bcell, K* ucell, int32_t* ustart, int32_t* cbox,
                      int32_t* ctab, uint32_t* nbox_dev, uint32_t* ncells_dev, hipStream_t s);

// btight[b]: bit 0 tight, bit 1 tight with >= minPts rows, bit 2 in a cell
// that can hold cores (cell_core); *nloose counts boxes of two or more rows
// that are not tight, nlarge[0] boxes of more than `large` rows, nlarge[1] those
// whose pairs the union takes by parts
template <typename T, int D>
void launch_box_tight(const BoxArgs<T>& a, const uint8_t* cell_core, uint8_t* btight,
                      unsigned int* nloose, int32_t large, unsigned int* nlarge, hipStream_t s);

// Components of the boxes with cores:
//   launch_list_boxes    list of the boxes with cores, *count += their
//                        number; bparent and cmin (of launch_box_clusters)
//                        reset
//   launch_box_hook      hook forest over the listed boxes: every box points
//                        at some earlier box joined to it
//   launch_box_roots     root of every box -> rsnap (-1 without cores), the
//                        roots to list (when not null), *count += their number
//   launch_box_root_join every listed root joins the first tree of another
//                        box it meets (one round: a second one costs more than
//                        the union then saves, 30k of 6 doubles 599 -> 637 us,
//                        100k of 3 floats 324 -> 340); then launch_box_roots
//   launch_box_union     (list: scratch for the boxes, out of the *nblist of
//                        blist, of those of the m cells that can have open
//                        pairs, *nlist += their number) the pairs still open (different trees in rsnap,
//                        within eps by their bounding boxes; *nopen += their
//                        number), every one decided exactly (large: boxes of
//                        launch_box_tight's nlarge[1] may exist)
//   then launch_box_clusters.
// List lengths stay on the device (kernels of persistent grids).  heavy
// holds heavy_cap entries of scratch; *nheavy, *nopen and every count are
// zeroed by the caller.
void launch_list_boxes(Count nbox, const int32_t* bmincore, int32_t* list, unsigned int* count,
                       int32_t* bparent, unsigned long long* cmin, hipStream_t s);
template <typename T, int D>
void launch_box_hook(const BoxArgs<T>& a, const uint32_t* roff, const int2* rboxes,
                     const int32_t* bmincore, const uint8_t* core, const int32_t* blist,
                     const unsigned int* nlist, int32_t* bparent, hipStream_t s);
void launch_box_roots(Count nbox, const int32_t* bmincore, int32_t* bparent, int32_t* rsnap,
                      int32_t* list, unsigned int* count, hipStream_t s);
template <typename T, int D>
void launch_box_root_join(const BoxArgs<T>& a, const uint32_t* roff, const int2* rboxes,
                          const int32_t* rsnap, const uint8_t* core, const int32_t* roots,
                          const unsigned int* nroots, int32_t* bparent, hipStream_t s);
template <typename T, int D>
void launch_box_union(const BoxArgs<T>& a, const uint32_t* roff, const int2* rboxes,
                      const int32_t* rsnap, const uint8_t* core, const int32_t* blist,
                      const unsigned int* nblist, Count m, int32_t* list, unsigned int* nlist,
                      const int32_t* box_of_slot, int2* heavy,
                      unsigned long long* nheavy, unsigned long long heavy_cap, int32_t* bparent,
                      unsigned long long* nopen, bool large, hipStream_t s);
// core[s] = 1 for the rows of tight boxes with >= minPts rows (btight bit 1),
// 0 for every other row; bmincore[b] = inrow[bstart[b]] for those boxes
// (every row is core and a box holds its rows in input order), INT_MAX for
// the others; rows[..] = the chunks of up to `chunk` (a power of two) rows of
// those other boxes whose cell can hold cores (btight bit 2), as (first slot,
// cell), *nrows += their number
void launch_core_init(int64_t n, const int32_t* box_of_slot, const uint8_t* btight,
                      const int32_t* bstart, const int32_t* bcell, const uint32_t* inrow,
                      uint8_t* core, int32_t* bmincore, int2* rows, unsigned int* nrows,
                      int chunk, hipStream_t s);
// p[0, n) = v
void fill_i32(int32_t* p, int32_t v, int64_t n, hipStream_t s);

void launch_box_clusters(Count nbox, const int32_t* bmincore, const int32_t* bcell,
                         const int32_t* cbox, const int32_t* bstart, const uint32_t* inrow,
                         const int32_t* ustart, int32_t* bparent, unsigned long long* cmin,
                         int32_t* compmin, int32_t* bcluster, hipStream_t s);

// pos_of_slot[s] = sorted position of slot s (the reference's order: cell,
// then input row), by a stable radix sort of the slots by occupied cell in
// input order; keys_a / vals_a / keys_b / vals_b (n words each), hist and
// tmp are scratch sized as for radix_sort_pairs<uint32_t>
void launch_positions(int64_t n, int32_t m, const int32_t* box_of_slot, const int32_t* bcell,
                      const uint32_t* inrow, uint32_t* keys_a, uint32_t* vals_a, uint32_t* keys_b,
                      uint32_t* vals_b, uint32_t* hist, uint32_t* tmp, uint32_t* pos_of_slot,
                      hipStream_t s);
}  // namespace hpd
