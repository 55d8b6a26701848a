// The order in which a wave of gemv_rows_kernel (qmm_gemv_batch.hip) issues its loads, and
// how many may be outstanding when an item's copies are read.  Plain C++, so that a test
// can walk the same code on the host and count.
#pragma once

namespace qmm {

// Walks the K groups [g0, g1), g0 < g1, of kMG items (row groups) each through
//   load_raw(g)          issue the loads of group g's weights (one register set)
//   convert()            wait for the weights loaded last and convert them
//   copy(g, mg, slot)    issue item (g, mg)'s copies into LDS slot 0 or 1
//   item(mg, slot, raws, next_g, next_mg)
//                        wait until at most one item's copies and `raws` groups' weight loads
//                        are outstanding, read the item in `slot`, issue item (next_g,
//                        next_mg)'s copies into it and compute
//   finish()             wait for everything; the weights loaded last count as used, so that
//                        no load is dropped as dead and the counts hold in the last group
// Items are copied two ahead, weights loaded one group ahead; loads past the slice's end
// repeat its last group and are not consumed.  The wait counts are those of the loop's own
// order, so the loads before the loop are issued in that order too: with one item per group
// a group's copies go before its weights, otherwise after them.
template <int kMG, class LoadRaw, class Convert, class Copy, class Item, class Finish>
__host__ __device__ __forceinline__ void walk_rows(int g0, int g1, LoadRaw load_raw, Convert convert, Copy copy,
                                                   Item item, Finish finish) {
    static_assert(kMG == 1 || kMG % 2 == 0, "the items of a K group start in slot 0, or alternate");
    auto at_most = [&](int g) { return g < g1 - 1 ? g : g1 - 1; };
    if constexpr (kMG == 1) {
        copy(g0, 0, 0);
        load_raw(g0);
        copy(at_most(g0 + 1), 0, 1);
    } else {
        load_raw(g0);
        copy(g0, 0, 0);
        copy(g0, 1, 1);
    }
    auto group = [&](int g, int par) {  // its first item in slot `par`
        convert();
        load_raw(at_most(g + 1));
#pragma unroll
        for (int mg = 0; mg < kMG; ++mg)  // the item two ahead: group g + (mg + 2) / kMG
            item(mg, (par + mg) & 1, kMG == 1 ? 2 : mg < 2 ? 1 : 0, at_most(g + (mg + 2) / kMG), (mg + 2) % kMG);
    };
    if constexpr (kMG == 1) {
        int g = g0;
        for (; g + 1 < g1; g += 2) {
            group(g, 0);
            group(g + 1, 1);
        }
        if (g < g1) group(g, 0);
    } else {
        for (int g = g0; g < g1; ++g) group(g, 0);
    }
    finish();
}

}  // namespace qmm
