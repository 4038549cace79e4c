// Launch shape of the level-1 updates (host only, no HIP dependency), shared by
// level1.hip and the CPU test that counts its idle lanes.
#pragma once

#include <algorithm>
#include <cstdint>

namespace hcb {

constexpr int kLevel1Threads = 256;
// Largest grid of the level-1 elementwise kernels (they grid-stride beyond).
constexpr int kMaxReduceBlocks = 1 << 21;

// Workgroups for a flat range of work items.
inline int full_grid(int64_t work_items) {
  const int64_t g = (work_items + kLevel1Threads - 1) / kLevel1Threads;
  return (int)std::max<int64_t>(1, std::min<int64_t>(g, kMaxReduceBlocks));
}

// Grid of an update at other increments or batch strides. rows: grid y walks the
// batch and x a vector, without a division per element; else x walks the flat
// index of all elements. Rows where they fill three quarters of their lanes:
// SAXPY of a batch, rows and flat, 100000 vectors of 16 31.8 and 6.5 us, of 128
// 33.6 and 28.9, of 200 42.3 and 42.8; 60000 of 256 32.5 and 33.7, of 300 55.4
// and 38.8; 20000 of 1000 41.5 and 45.7.
struct StridedGrid {
  bool rows;
  int x, y;
};
inline StridedGrid plan_strided(int64_t n, int64_t batch) {
  const int x = full_grid(n);
  if (batch == 1 || 4 * n >= 3 * (int64_t)x * kLevel1Threads)
    return {true, x, (int)std::min<int64_t>(batch, 65535)};
  return {false, full_grid(n * batch), 1};
}

}  // namespace hcb
