// Host side of the pivot panels' launch plan that needs no device: where the fronts of a level keep their
// scratch.
#pragma once
#include <cstdint>
#include <vector>

namespace sds {

// a front's scratch starts at a multiple of this many entries; the tasks hold the multiple, so that 32
// bits reach 2^37 entries
constexpr int PANEL_SCR_UNIT = 64;

// the offsets (in units) of fronts with the given entries of scratch each, and the level's entries in all;
// false if these are more than `limit`: the level then takes one pivot per launch pair, which needs none
inline bool panel_offsets(const std::vector<int64_t>& entries, int64_t limit, std::vector<int32_t>& off,
                          int64_t& total) {
    off.clear();
    total = 0;
    int64_t units = 0;
    for (int64_t e : entries) {
        if (units > INT32_MAX) return false;
        off.push_back((int32_t)units);
        units += (e + PANEL_SCR_UNIT - 1) / PANEL_SCR_UNIT;
        total = units * PANEL_SCR_UNIT;
        if (total > limit) return false;
    }
    return true;
}

}  // namespace sds
