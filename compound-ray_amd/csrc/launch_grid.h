// Grid sizes of launches whose work may exceed one grid (host code).
#pragma once

#include <stdint.h>

#include <algorithm>

namespace eye {

// HIP launches fewer than 2^32 threads along x: with workgroups of one wave,
// 67,108,863 of them.
constexpr uint64_t max_grid(int threads) { return 0xffffffffull / (uint64_t)threads; }

// The unit renderer's grid: `blocks` workgroups of work, each `threads` / 64
// grabs, over which a grid of `grid` workgroups strides (all of them where they
// fit one grid).  fixed: blocks of 256 threads as asked for, 0 for a workgroup
// each.
struct UnitGrid {
  uint32_t blocks;
  uint32_t grid;
};
inline UnitGrid unit_grid(uint64_t units, int units_per_grab, int threads, int fixed) {
  const uint64_t per_block = (uint64_t)units_per_grab * (uint64_t)(threads / 64);
  const uint64_t blocks = (units + per_block - 1) / per_block;
  const uint64_t asked = fixed > 0 ? (uint64_t)fixed * (uint64_t)(256 / threads) : blocks;
  const uint64_t stride = std::min<uint64_t>(max_grid(threads), 0x100000000ull - blocks);
  return UnitGrid{(uint32_t)blocks, (uint32_t)std::min(std::min(asked, blocks), stride)};
}

}  // namespace eye
