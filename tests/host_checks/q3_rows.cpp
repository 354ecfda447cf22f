// Every entry the order-3 kernel reads in the rows above its tile lies in its
// row, and every (L, k) is visited exactly once: the walk of q3.hip with the
// helpers it uses.  Prints what is wrong and returns 1.
#include <cstdio>
#include <map>
#include <utility>

#include "q3_rows.h"

using namespace mlip;

int main() {
    int bad = 0;
    for (int lq = 0; lq <= 10; ++lq)
        for (int maxl = lq; maxl <= 20; ++maxl) {
            const int levels = q3_rows_above(lq, maxl), share = q3_row_share(lq, levels);
            std::map<std::pair<int, int>, int> seen;
            auto read = [&](int L, int k) {
                const int at = L * (L + 1) / 2 + L - k;
                if (k >= 0 && at >= L * (L + 1) / 2 && at < n_lmh_of(maxl)) return;
                std::printf("lmaxq3 %d maxl %d: row %d entry %d read\n", lq, maxl, L, k);
                ++bad;
            };
            for (int wave = 0; wave < kWavesPerWg; ++wave)
                for (int it = wave; it < levels * share; it += kWavesPerWg) {
                    const int L = q3_row_level(it, share, lq);
                    int k = q3_row_first(it, share);
                    read(L, k);
                    for (; k <= L; k += share) {
                        read(L, k + share < L ? k + share : L);
                        ++seen[{L, k}];
                    }
                }
            for (int L = lq + 1; L <= maxl && L <= kMaxLQ12; ++L)
                for (int k = 0; k <= L; ++k)
                    if (seen[{L, k}] != 1) {
                        std::printf("lmaxq3 %d maxl %d: (%d, %d) visited %d times\n", lq, maxl, L, k, seen[{L, k}]);
                        ++bad;
                    }
        }
    return bad ? 1 : 0;
}
