// Cells: the distinct (m, k, n) of a mode set and the modes in each.
//
// Modes that differ only in l share their phase m Phi_phi + k Phi_theta +
// n Phi_r, and everything else of the mode sum is linear in the amplitudes, so
// a direct sum needs one phase (and one sincos) per cell instead of one per
// mode: the 3843 modes of the l <= 10, |n| <= 30 set have 671 cells.
#pragma once

#include "few_common.hpp"

namespace few {

// Cells in order of their first mode; cell c holds the modes
// member[start[c]] .. member[start[c + 1] - 1], ascending.  start == nullptr:
// no grouping, cell c is mode c.
struct CellIndex {
    const int *count = nullptr;   // number of cells
    const int *start = nullptr;
    const int *member = nullptr;
};

// Mode sets below this size are not grouped: the two launches of the index
// (5 us at 64 modes, 8 at 500, 23 at 3843) cost more than the few shared phases of a
// small set save.
constexpr int CELL_MIN_MODES = 64;

// Device workspace of the index of K modes.
size_t cell_index_bytes(int K);

// Builds the index in `ws` (cell_index_bytes(K) bytes; two launches, no
// synchronisation).  rows (optional): two int arrays of `width` values per mode,
// which the modes of one cell must share as well.
int launch_cell_index(const int *m, const int *k, const int *n, int K, const int *row_a,
                      const int *row_b, int width, void *ws, CellIndex &out, hipStream_t stream);

}  // namespace few
