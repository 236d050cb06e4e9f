// The order of the correction's windows of z-layer tiles (plain C++: the kernel
// and host programs use the same rule).
#pragma once
#include <cstdint>

namespace gg {
// Workgroups take the positions u = 0, 1, 2, ... in turn, and workgroup b runs
// on XCD b % 8, so a position's XCD is u mod 8: each eight consecutive windows
// go one to each XCD.  Boxes of equal sides in a row repeat the same work every
// few windows (a box of side 32 has four windows of eight layers, the first and
// the last with little of the band), so the eight windows of position group
// u / 8 are rotated by a golden-ratio hash of the group.  A bijection on every
// multiple of eight.
constexpr int run_window(int u) {
  const uint32_t turn = ((uint32_t)u >> 3) * 2654435769u >> 29;
  return (int)(((uint32_t)u & ~7u) | (((uint32_t)u + turn) & 7u));
}
}  // namespace gg
