// The prefill GEMM's launch shapes and the rule that picks one (qmm_gemm.hip).  Plain C++, so
// that a test can ask on the host.
#pragma once
#include <cstdint>

#include "openmini_qmm.h"

namespace qmm {

// Workgroups as column slices x K parts of waves, and 16-column weight tiles per wave:
//   0: 128 x 192, 4 x 2 waves, 3 tiles   4: 64 x 64, 2 x 4 waves, 2 tiles
//   1: 128 x 128, 4 x 2 waves, 2 tiles   5: 64 x 32, 1 x 8 waves, 2 tiles
//   2:  64 x  96, 2 x 4 waves, 3 tiles   6: 64 x 64, 2 x 2 waves, 2 tiles
//   3:  64 x 128, 4 x 2 waves, 2 tiles   7: 128 x 96, 2 x 2 waves, 3 tiles
constexpr int kShapes = 8;
constexpr int kShapeRows[kShapes] = {128, 128, 64, 64, 64, 64, 64, 128};
constexpr int kShapeTiles[kShapes] = {12, 8, 6, 8, 4, 2, 4, 6};  // weight tiles (16 columns) per workgroup

// Few and large workgroups leave CUs idle or a last round part-filled; small ones cost more
// per flop (each B fragment serves fewer MFMAs, each A fragment fewer tiles).  The model:
// workgroups run in rounds of 256 CUs x as many as share one; a round costs a start (first
// loads, K-part sums, stores) and a time per K element, a last round of j workgroups per CU
// that of j.  Fitted to every shape forced at 27 weight shapes x 64 .. 2048 rows for Q4_0,
// Q8_0, Q4_K and Q6_K each, and at larger ones: over the 3430 of the sweep the pick is on
// average 0.1% slower than the fastest shape, at 28 of them by more than 3% and at most by 8%;
// with weights that come from HBM 0.1%, 30 of 1740, 9%.
// Types have rows of their own where their kernels' times differ: one row for Q4_0, Q8_0 and
// Q4_K picked shapes up to 21% slower than the fastest for Q8_0 (fp32 x, 11008 x 2048 at 384
// rows: 64.1 us against 53.0).  Shapes 6 and 7, four waves with two to four workgroups on a
// CU, are there for the sizes between two rounds of the large tiles: bf16 x, Q8_0 11008 x 4096
// at 768 rows 122 us without them, 114 in shape 6, 110 in shape 7; 13824 x 4096 at 100 rows
// 33.1 -> 30.1 in shape 6, at 1536 rows 244 -> 228 in shape 7.
// (Long runs.  In the first milliseconds after idle the card is slower and small tiles lose
// more: where Q6_K on bf16 x tied in long runs, 11008 x 4096 at 512 rows 121 us in shapes 1 and
// 6 but 141 and 154 after idle, shape 6's row is priced 1.5% up.)
// Left: a launch that fills its CUs exactly once with two or more workgroups each takes up to
// 13% longer on split x than the model says (part-filled ones are right, and with weights from
// HBM the pick still wins): 16306 x 2816 at 109 rows 35.9 us in shape 4, 32.8 in shape 3.
struct ShapeCost {
    double start = 0.0;                 // us of a round
    double per_k[4] = {0., 0., 0., 0.}; // us of a round per 1000 K elements, 1 .. 4 workgroups on a CU
};

// per_cu: workgroups of each shape's kernel that one CU holds; below 0 where it is not built.
// Fixed per shape, so a row's bits depend only on m and the weight.
inline int choose_gemm_shape(int type, int64_t n_tiles, int64_t k, int64_t m, const int (&per_cu)[kShapes], bool split_x) {
    static const ShapeCost kCost[6][kShapes] = {
        // bf16 x: Q4_0, Q4_K
        {{5.6, {12.7}}, {3.7, {8.95}}, {2.1, {4.42}}, {2.2, {5.70, 9.72}},
         {1.4, {3.16, 5.47}}, {1.6, {1.68}}, {1.2, {4.26, 6.06, 8.35, 10.5}}, {4.1, {8.40, 12.9}}},
        // bf16 x: Q8_0
        {{6.4, {13.4}}, {4.1, {9.28}}, {2.6, {4.89}}, {2.8, {6.06, 10.5}},
         {1.7, {3.46}}, {1.8, {1.92}}, {1.3, {4.39, 6.35, 8.66}}, {4.6, {10.1, 14.6}}},
        // bf16 x: Q6_K (0, 3 and 7 not built)
        {{}, {4.1, {13.6}}, {3.1, {7.44}}, {},
         {2.0, {5.19}}, {2.1, {2.61}}, {1.6, {6.60, 9.45}}, {}},
        // split x: Q4_0, Q4_K
        {{6.5, {18.9}}, {4.3, {13.7}}, {2.4, {6.25}}, {1.8, {8.37, 13.9}},
         {0.7, {5.34, 8.31}}, {1.3, {2.99}}, {1.3, {7.07, 8.87, 12.4, 16.0}}, {4.7, {13.8, 20.9}}},
        // split x: Q8_0
        {{5.2, {20.3}}, {4.5, {14.5}}, {3.1, {7.07}}, {1.6, {9.00, 15.0}},
         {1.0, {5.64, 8.94}}, {1.5, {3.19}}, {1.4, {7.49, 9.32, 13.4, 17.3}}, {4.6, {14.4, 21.5}}},
        // split x: Q6_K
        {{5.7, {32.0}}, {4.2, {22.6}}, {3.2, {10.6}}, {2.4, {14.0}},
         {1.6, {7.61}}, {2.4, {4.08}}, {1.8, {9.94, 14.2, 20.0}}, {4.7, {22.0, 33.8}}},
    };
    constexpr int64_t kCus = 256;
    const int kind = type == OPENMINI_QMM_Q8_0 ? 1 : type == OPENMINI_QMM_Q6_K ? 2 : 0;
    const ShapeCost* cost = kCost[(split_x ? 3 : 0) + kind];
    int best = -1;
    double best_us = 0.0;
    for (int i = 0; i < kShapes; ++i) {
        if (per_cu[i] < 0 || cost[i].start == 0.0) continue;
        const int64_t wgs = (n_tiles + kShapeTiles[i] - 1) / kShapeTiles[i] * ((m + kShapeRows[i] - 1) / kShapeRows[i]);
        int share = 1;  // workgroups on a CU
        while (share < 4 && share < per_cu[i] && cost[i].per_k[share] > 0.0) ++share;
        const int64_t slots = share * kCus, full = wgs / slots, left = wgs % slots;
        double per_k = (double)full * cost[i].per_k[share - 1];
        if (left) per_k += cost[i].per_k[(left + kCus - 1) / kCus - 1];
        const double us = (double)(full + (left ? 1 : 0)) * cost[i].start + per_k * 0.001 * (double)k;
        if (best < 0 || us < best_us) best = i, best_us = us;
    }
    return best;
}

}  // namespace qmm
