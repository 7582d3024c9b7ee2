// Launches of any number of workgroups: a HIP grid holds fewer than 2^32 work-items, so larger ones are split.
// Host code only (no HIP headers).
#pragma once

#include <cstddef>
#include <cstdint>

namespace oct {

// workgroups of `threads` work-items that one launch can hold
constexpr size_t grid_limit(size_t threads) { return 0xffffffffull / threads; }

// launch(first workgroup, workgroups) for the ranges of at most grid_limit that make up `blocks`
template <class F>
inline void for_grids(size_t blocks, size_t threads, F &&launch) {
    for (size_t at = 0; at < blocks; at += grid_limit(threads)) {
        const size_t left = blocks - at;
        launch((uint32_t)at, (unsigned)(left < grid_limit(threads) ? left : grid_limit(threads)));
    }
}

}  // namespace oct
