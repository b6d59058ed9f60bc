// box_levels.hpp -- where the build's table of aligned unions keeps its levels.  Plain C++: the host and the device use it.
//
// Level k holds the unions of 2^k aligned leaf slots, whole ones only; the levels 1, 2, ... lie one behind the other and
// take fewer than n boxes in all.
#pragma once

#include <cstdint>

namespace rtgpu {

// (up to 2^27 leaves the last launch of eight levels reaches level 32, beyond a shift's range)
constexpr uint32_t box_count(uint32_t n, uint32_t level) { return level < 32u ? n >> level : 0u; }

// where level k begins, k >= 1
constexpr uint64_t boxes_before(uint32_t n, uint32_t k) {
    uint64_t s = 0;
    for (uint32_t l = 1; l < k; ++l) s += box_count(n, l);
    return s;
}

}  // namespace rtgpu
