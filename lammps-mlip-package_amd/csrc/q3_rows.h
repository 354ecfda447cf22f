// Walk of the adjoint rows above the order-3 kernel's tile (q3.hip): levels L =
// lmaxq3 + 1 .. min(maxl, kMaxLQ12), the entries m = -k of a level dealt over
// `share` waves.  Item `it` (one wave's) takes k = q3_row_first, + share, ... up
// to L of its level.  A level has at least lmaxq3 + 2 entries, and no more waves
// share one: every item's first entry lies in its row, so the kernel may read it
// before it tests for the row's end.
#pragma once

#include "model.h"

namespace mlip {

constexpr int q3_rows_above(int lmaxq3, int maxl) { return (maxl < kMaxLQ12 ? maxl : kMaxLQ12) - lmaxq3; }
constexpr int q3_row_share(int lmaxq3, int levels) {
    const int waves = levels > 0 ? (kWavesPerWg + levels - 1) / levels : 1;
    return waves < lmaxq3 + 2 ? waves : lmaxq3 + 2;
}
constexpr int q3_row_level(int it, int share, int lmaxq3) { return lmaxq3 + 1 + it / share; }
constexpr int q3_row_first(int it, int share) { return it % share; }

}  // namespace mlip
