// What the lists of a LAMMPS call keep: everything while calls stay alike, at most
// four times what the last call used (small arrays aside) after larger ones.
#include <cstdio>

#include "lammps_lists.h"

static void call(LammpsLists& L, size_t atoms, size_t pairs, bool half) {
    L.local_of_tag.clear();
    L.x.resize(3 * atoms);
    for (auto* v : {&L.elem, &L.elem_own, &L.poff, &L.gof, &L.owner_of_local, &L.fill}) v->resize(atoms + 1);
    for (auto* v : {&L.pnbr, &L.pcen}) v->resize(pairs);
    L.gen.resize(2 * pairs);
    if (half) L.local_of_tag.resize(4 * atoms);
    L.trim();
}

int main() {
    LammpsLists L;
    call(L, 100000, 10000000, true);
    const size_t big = L.held();
    const int32_t* at = L.pnbr.data();
    call(L, 90000, 9000000, true);
    if (L.held() != big || L.pnbr.data() != at) return std::printf("given back between calls alike\n"), 1;
    call(L, 100000, 1000000, false);
    const size_t used = 24 * 100000 + 6 * 4 * 100001 + 16 * 1000000, small = 11 * LammpsLists::kSmall * 8;
    if (L.held() > LammpsLists::kSpare * used + small || !L.local_of_tag.empty())
        return std::printf("%zu bytes kept of %zu for a call of %zu\n", L.held(), big, used), 1;
    call(L, 10, 20, true);
    if (L.held() > small) return std::printf("%zu bytes kept after a small call\n", L.held()), 1;
    return 0;
}
