// Memory shared between the groups of a convolution batch (host code only).
#pragma once

#include <algorithm>
#include <cstddef>
#include <cstdint>
#include <vector>

namespace s2 {

// Bytes [lo, hi) that a group reads or writes.
struct MemRange {
    uintptr_t lo, hi;
    int group;
    bool write;
};

// Whether some group writes bytes that another group reads or writes: such
// groups depend on the order they run in.  One sweep over the ranges by start,
// with the furthest end so far, its group, and the furthest end of any other
// group, over all ranges and over the written ones.
inline bool groups_conflict(std::vector<MemRange> v) {
    struct Ends {
        uintptr_t best = 0, other = 0;
        int group = -1;
        uintptr_t beside(int g) const { return g == group ? other : best; }
        void add(uintptr_t hi, int g) {
            if (g == group) {
                best = std::max(best, hi);
            } else if (hi > best) {
                other = best;
                best = hi;
                group = g;
            } else {
                other = std::max(other, hi);
            }
        }
    } all, written;
    std::sort(v.begin(), v.end(), [](const MemRange& a, const MemRange& b) { return a.lo < b.lo; });
    for (const MemRange& r : v) {
        if (r.lo >= r.hi) continue;
        if ((r.write ? all : written).beside(r.group) > r.lo) return true;
        all.add(r.hi, r.group);
        if (r.write) written.add(r.hi, r.group);
    }
    return false;
}

}  // namespace s2
