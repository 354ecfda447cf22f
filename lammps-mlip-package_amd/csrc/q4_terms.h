// Products of three variables that order-4 adjoint rows l <= 2 are made of, in
// the order the kernel (q3.hip) and the host tables (model.cpp) walk them.
// Variable v = species * 9 + l (l + 1) + m, l <= 2; products i <= j <= k whose m sum
// M lies in 0..2 reach the outputs (L, m = -M) with L >= M and even l sum.
// Coefficients follow as [part][pair (i, j)][k][L][S], pair p of a model's used
// pairs belonging to part p mod kQ4Parts.
#pragma once

namespace mlip {

constexpr int kQ4Parts = 4;

constexpr int q4_l(int v) { return v % 9 == 0 ? 0 : v % 9 < 4 ? 1 : 2; }
constexpr int q4_m(int v) { return v % 9 - q4_l(v) * (q4_l(v) + 1); }
constexpr int q4_outputs(int i, int j, int k) {
    const int M = q4_m(i) + q4_m(j) + q4_m(k), par = (q4_l(i) + q4_l(j) + q4_l(k)) & 1;
    if (M < 0 || M > 2) return 0;
    int n = 0;
    for (int L = M; L < 3; ++L) n += (L & 1) == par;
    return n;
}
constexpr bool q4_used(int i, int j, int k) { return q4_outputs(i, j, k) > 0; }
constexpr bool q4_pair_used(int nt, int i, int j) {
    for (int k = j; k < 9 * nt; ++k)
        if (q4_used(i, j, k)) return true;
    return false;
}
// coefficients of parts 0 .. part - 1
constexpr int q4_count_parts(int nt, int part) {
    int pair = 0, n = 0;
    for (int i = 0; i < 9 * nt; ++i)
        for (int j = i; j < 9 * nt; ++j) {
            if (!q4_pair_used(nt, i, j)) continue;
            if (pair++ % kQ4Parts >= part) continue;
            for (int k = j; k < 9 * nt; ++k) n += q4_outputs(i, j, k) * nt;
        }
    return n;
}
constexpr int kQ4Offset[2][kQ4Parts + 1] = {
    {0, q4_count_parts(1, 1), q4_count_parts(1, 2), q4_count_parts(1, 3), q4_count_parts(1, 4)},
    {0, q4_count_parts(2, 1), q4_count_parts(2, 2), q4_count_parts(2, 3), q4_count_parts(2, 4)}};
constexpr int q4_offset(int nt, int part) {
    return part == 0 ? 0 : part == 1 ? kQ4Offset[nt - 1][1] : part == 2 ? kQ4Offset[nt - 1][2] : kQ4Offset[nt - 1][3];
}
constexpr int q4_total(int nt) { return kQ4Offset[nt - 1][kQ4Parts]; }

}  // namespace mlip
