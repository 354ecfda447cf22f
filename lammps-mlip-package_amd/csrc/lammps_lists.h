// A LAMMPS-shaped neighbor list as the engine's pair and gather lists.
#pragma once

#include <cstddef>
#include <cstdint>
#include <vector>

// Kept in the context from call to call for its memory: fresh vectors of a few
// megabytes are page faults on every call.  What is kept follows the calls: after
// each one trim() gives back arrays more than kSpare times what it needed, and a
// context that takes a resident structure, a batch or a pool keeps nothing.
struct LammpsLists {
    int nall = 0;
    int64_t npairs = 0;
    std::vector<double> x;
    std::vector<int32_t> elem, elem_own, poff, pnbr, pcen, gof, gen;
    std::vector<int32_t> owner_of_local, local_of_tag, fill;  // work space

    static constexpr size_t kSpare = 4;
    static constexpr size_t kSmall = 1 << 16;  // entries not worth giving back

    void trim() {
        trim(x);
        for (std::vector<int32_t>* v : {&elem, &elem_own, &poff, &pnbr, &pcen, &gof, &gen, &owner_of_local,
                                        &local_of_tag, &fill})
            trim(*v);
    }
    size_t held() const {  // bytes
        size_t n = 0;
        for (const std::vector<int32_t>* v : {&elem, &elem_own, &poff, &pnbr, &pcen, &gof, &gen, &owner_of_local,
                                              &local_of_tag, &fill})
            n += v->capacity() * sizeof(int32_t);
        return n + x.capacity() * sizeof(double);
    }

private:
    template <typename T>
    static void trim(std::vector<T>& v) {
        if (v.capacity() > kSmall && v.capacity() / kSpare > v.size()) std::vector<T>(v).swap(v);
    }
};
