// qm_linear_rows_params.h — launch parameters shared by the two kernels behind qm_linear_rows / qm_gate_up_swiglu_rows.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace qm {

constexpr int kRowsGroups = 5;

struct LinearRowsParams {
    const uint16_t* input;        // [rows][reduction]
    const uint16_t* weight[2];    // [columns][reduction]; [1] = the up matrix (DUAL)
    const uint16_t* bias;         // [columns] or NULL
    const uint16_t* residual;     // [rows][columns] or NULL
    uint16_t* output;             // [rows][columns]
    int rows, columns, reduction;
    int columns_per_block;        // 8 or 4 (4: the two halves of the block take four token rows each)
    // (matrix cores, few token rows) the reduction cut into reduction_parts pieces, one block each: the fp32 sums of
    // piece z go to partials[z] ([rows][columns]; a gate/up pair: gate plane, then up plane) and a second launch adds the
    // pieces in order and rounds.  1: every block takes the whole reduction and rounds its sums itself.
    int reduction_parts;
    float* partials;
    // (matrix cores, no gate/up pair) up to kRowsGroups linears of the same input in one grid: the column tiles of linear g
    // start at tile group_first_tile[g] (group 0 at 0), and a block of group g > 0 takes weight / bias / output / columns
    // from group_*[g - 1] instead of the fields above.  groups = 1: one linear.
    int groups;
    int group_first_tile[kRowsGroups - 1];
    const uint16_t* group_weight[kRowsGroups - 1];
    const uint16_t* group_bias[kRowsGroups - 1];
    uint16_t* group_output[kRowsGroups - 1];
    int group_columns[kRowsGroups - 1];
    // (matrix cores, no gate/up pair, reduction uncut) sums != NULL: the fp32 sums as they are go to sums /
    // group_sums[g - 1] ([rows][columns] floats) and nothing to the outputs; bias and residual are not read.
    float* sums;
    float* group_sums[kRowsGroups - 1];
    // a linear of its own input and reduction (a multiple of 128 as well): NULL / 0 = the first one's
    const uint16_t* group_input[kRowsGroups - 1];
    int group_reduction[kRowsGroups - 1];
    // elements from a row of input and weights to the next, where a linear takes a piece of longer rows; 0: its reduction
    int pitch, group_pitch[kRowsGroups - 1];
    // blocks in the order linear by linear (all row tiles of the first, then of the next) instead of row tile by row
    // tile: the linears with the long reductions first, so that none of them starts late
    int linear_by_linear;
    // (matrix cores, reduction uncut, one linear or pair) several matrices of one shape, one behind the other: row tile t of
    // tile_rows rows (64 or 128) takes matrix tile_matrix[t], or is left out where that is negative
    const int32_t* tile_matrix;
    int tile_rows;
    // (a cut reduction of 1024 or 2048 columns) norm_weight != NULL: the launch that adds the pieces also leaves RMSNorm of the output's rows
    const uint16_t* norm_weight;
    uint16_t* normalized;
    float epsilon;
    // (a cut reduction) 128 x 128 tiles
    bool wide_tiles;
};

// The grid's width for so many column tiles, by row tiles and pieces of the reduction.  Blocks go to the eight dies of 32 CUs in turn, one to a CU:
// where 8 divides the width, the row tiles of a column read its weights on one die, but the dies with a column more may walk a round of blocks more
// than all of them do when the tiles are dealt out one by one.  Rounded up (the blocks beyond end at once) a grid takes, of its time as it is, reductions
// of 1024 and 2048, weights in the caches and from memory: with more than forty columns 0.57 to 1.00 where the rounds stay the same, 0.83 to 0.95 where
// three or more become one more, 0.93 to 1.18 where two become three and 0.90 to 1.71 where one becomes two; with fewer columns 0.60 to 1.21 even where
// the rounds stay the same.  (us: 1024 tokens, 81 columns by 8 row tiles of 2048 64.8 -> 56.1; 130 tokens, 84 by 3 of 1024 7.4 -> 11.0.)
inline int rows_grid_columns(int column_tiles, int row_tiles, int pieces) {
    const int64_t rounded = (column_tiles + 7) / 8 * 8, rows = static_cast<int64_t>(row_tiles) * pieces;
    const int64_t busiest = (rounded / 8 * rows + 31) / 32, even = ((column_tiles * rows + 7) / 8 + 31) / 32;
    return column_tiles > 40 && row_tiles > 1 && 3 * busiest <= 4 * even ? static_cast<int>(rounded) : column_tiles;
}

// Whether tiles of `tile_columns` columns and `step` k cover every linear exactly.  The kernel bounds token rows only: a tile that hangs over a linear's
// last column would read weight rows past the matrix (half a tile of 2048 inputs: 256 KiB, past the allocation as well) and write the
// columns it has too many over the next row, past the output in the last; a piece that is no whole number of steps would leave inputs out; planes of
// pieces are laid out for one linear, and the norm behind them takes two planes at a time of rows that 256 threads hold.
inline bool rows_are_whole_tiles(const LinearRowsParams& prm, int tile_columns, int step) {
    if (prm.rows <= 0 || prm.groups < 1 || prm.groups > kRowsGroups || prm.reduction_parts < 1) return false;
    int64_t before = 0;
    for (int g = 0; g < prm.groups; ++g) {
        const int columns = g == 0 ? prm.columns : prm.group_columns[g - 1];
        const int reduction = g == 0 || !prm.group_reduction[g - 1] ? prm.reduction : prm.group_reduction[g - 1];
        if (columns <= 0 || columns % 128 || columns % tile_columns) return false;
        if (reduction <= 0 || reduction % 128 || reduction % (static_cast<int64_t>(step) * prm.reduction_parts)) return false;
        if (g > 0 && prm.group_first_tile[g - 1] != before / 128) return false;
        before += columns;
    }
    if (prm.reduction_parts == 1) return true;
    return prm.groups == 1 && prm.partials && (!prm.norm_weight || (prm.reduction_parts % 2 == 0 && (prm.columns == 1024 || prm.columns == 2048)));
}

// The row linears on the matrix cores (qm_linear_rows_mfma.hip).  `dual`: weight[0] / weight[1] are the gate and up
// matrices and the epilogue is SwiGLU.  Columns and reductions that are not multiples of 128: QM_ERR_GEOMETRY, nothing is launched.
int32_t launch_rows_mfma(const LinearRowsParams& prm, bool dual, hipStream_t stream);

// Into how many pieces launch_rows_mfma cuts the reduction when it is given a workspace for the partial sums (a pure
// function of the shape), and the bytes that workspace must hold (0: the shape is not cut).
int rows_mfma_reduction_parts(int rows, int columns, int reduction, bool dual);
size_t rows_mfma_workspace_bytes(int rows, int columns, int reduction, bool dual);
// The same where the pieces are added by the launch of a norm that is there anyway; *wide: in 128 x 128 tiles.
int rows_mfma_norm_parts(int rows, int columns, int reduction, bool* wide);

}  // namespace qm
