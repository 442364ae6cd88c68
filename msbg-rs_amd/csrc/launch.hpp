// Host-side limits of a kernel launch.
#pragma once

#include <cstdint>

namespace msbg {

// The most work-groups of `threads` lanes that a launch may have along an axis:
// HIP refuses 2^32 lanes and more.
constexpr int64_t max_groups(int threads) { return (((int64_t)1 << 32) - 1) / threads; }

}  // namespace msbg
