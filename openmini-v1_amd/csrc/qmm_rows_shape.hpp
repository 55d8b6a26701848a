// Which batched calls of more than 16 rows run as one pass over the weight (gemv_rows_kernel,
// qmm_gemv_batch.hip) and which as 16-row passes.  Plain C++, so that a test can ask on the
// host.
#pragma once
#include <cstdint>

#include "openmini_qmm.h"

namespace qmm {

constexpr int kPassRows = 16;             // rows of one row group, and of a pass of the 16-row kernel
constexpr int kRowsMax = 4 * kPassRows;   // most rows of one multi-row-group launch

// T row tiles and W K slices per workgroup of the multi-row-group launch.
struct RowsShape {
    int t = 1, w = 0;       // w = 0: 16-row passes only
    int least = kPassRows;  // it takes more rows than this
    int most = kRowsMax;    // and at most this many in one launch
    int groups = 0;         // the weight's K groups
    int limits = -1;        // its row of kOnePassGroups; -1: no limit
};

// Two-way splits with one tile per workgroup: one pass has half the workgroups of the 16-row
// passes.  That costs more the longer K is, more for a block minimum's sums and where the
// split's workgroups had CUs of their own (at most 128 tiles), and fewer saved passes pay for
// it where the last row group is part empty.  One pass from fewer K groups than this on,
// measured at 40 .. 126 groups of 1100 .. 4096 rows (16-row passes over one pass):
//   up to 128 tiles, Q4_0 17 rows 1.09 / 1.04 / 0.97 at 72 / 88 / 96 groups, 24 rows 1.10 /
//   1.02 / 0.98 at 88 / 96 / 112, 33 rows 1.04 / 1.00 / 0.98 at 96 / 112 / 126; Q8_0 0 - 6% and
//   Q6_K 4% below; Q4_1 and Q5_K, 17 rows 1.07 / 0.96 at 40 / 48, 24 rows 1.02 / 0.95 at 48 /
//   72, 32 rows 1.04 / 0.97 at 88 / 96, 40 rows 1.09 / 1.00 / 0.94 at 56 / 72 / 88, 64 rows
//   1.14 / 1.06 / 1.03 / 1.00 at 88 / 96 / 112 / 126;
//   129 - 256 tiles, Q4_1 17 rows 1.09 / 0.96 at 56 / 72, 24 rows 1.01 / 0.97 at 88 / 96, 40
//   rows 1.03 / 0.99 at 88 / 96, 56 rows 1.07 at 112; the others 0.98 or more everywhere.
constexpr int kOnePassGroups[3][9] = {
    // rows: 17-20, 21-24, 25-28, 29-32, 33-36, 37-40, 41-48, 49-56, 57-64
    {90, 96, 128, 128, 112, 128, 128, 128, 128},  // up to 128 tiles
    {46, 64, 78, 90, 68, 74, 88, 96, 124},        // the same with a block minimum
    {66, 92, 116, 128, 80, 94, 116, 128, 128},    // 129 - 256 tiles, Q4_1
};

// For a weight (or a pair) of n_tiles row tiles and `groups` K groups whose 16-row call runs
// `split` K splits of `waves` waves.  The waves cut K as a 16-row call's do, so a row has the
// same bits in either: its own wave count, or eight slices in place of a two-way split over
// four-wave workgroups.  Splits with more waves than that, and K of fewer than 8 groups (one
// wave), have no such form.  The other lines are where 16-row passes are faster (MI355X, us,
// 16-row passes -> one pass):
//   more than 768 row tiles: one pass holds at most 3 tiles per workgroup, 16-row passes up to
//     8, and the activation split is shared by fewer tiles than the saved passes win back
//     (28672 x 8192, 20 / 40 rows: 63 -> 75, 98 -> 109).  A pair, at one tile of each weight,
//     from 512 on (11008 x 4096, 20 / 40 rows: 32.3 -> 39.7, 50.3 -> 51.4) and up to two row
//     groups (Q5_K 8192 x 4096, 20 / 40 rows: 36.9 -> 39.8, 58.3 -> 49.9).
//   three tiles of a type with a block minimum in eight slices: four row groups do not fit the
//     registers (28-44 spilled; Q5_K 12288 x 8192, 40 rows: 82 -> 114), two do, with at most 8
//     spilled (32 rows: 57 -> 47; 40 rows in two launches 68).
//   two-way splits with one tile per workgroup: kOnePassGroups.
inline RowsShape rows_shape(int type, int64_t n_tiles, int64_t groups, int split, int waves, bool pair) {
    constexpr int64_t kCUs = 256;
    RowsShape r;
    const int64_t per_cu = (n_tiles + kCUs - 1) / kCUs;
    if (per_cu > (pair ? 2 : 3)) return r;
    if (split == 1 && waves >= 4)
        r.w = waves;
    else if (split == 2 && waves == 4)
        r.w = 8;
    r.t = pair ? 1 : (int)per_cu;
    r.groups = (int)groups;
    if (pair) r.least = 2 * kPassRows;
    const bool block_min = type == OPENMINI_QMM_Q4_1 || type == OPENMINI_QMM_Q5_K;
    if (block_min && r.t == 3 && r.w == 8) r.most = 2 * kPassRows;
    if (split == 2 && r.t == 1) r.limits = n_tiles <= kCUs / 2 ? (block_min ? 1 : 0) : type == OPENMINI_QMM_Q4_1 ? 2 : -1;
    return r;
}

// Rows of the next launch when `rest` are left: more than kPassRows, one multi-row-group
// launch; else one 16-row pass.
inline int next_rows(const RowsShape& r, int64_t rest) {
    bool many = r.w != 0 && rest > r.least;
    const int n = (int)(rest < r.most ? rest : r.most);
    if (many && r.limits >= 0) {
        const int at = n <= 40 ? (n - 17) / 4 : 6 + (n - 41) / 8;  // n in 17 .. 64
        many = r.groups < kOnePassGroups[r.limits][at];
    }
    return many ? n : n < kPassRows ? n : kPassRows;
}

}  // namespace qmm
