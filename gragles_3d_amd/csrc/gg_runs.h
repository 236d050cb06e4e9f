// The order of the correction's windows of z-layer tiles (plain C++: the kernel
// and host programs use the same rule).
#pragma once
#include <cstdint>

namespace gg {
// Windows in a row that go to one XCD, about a box of the kernel's class (sides
// up to nmax, windows of zt tiles): the runs of a grain then share that XCD's L2.
constexpr int run_chunk(int nmax, int zt) {
  int c = 1;
  while (2 * c * zt <= nmax) c *= 2;
  return c;
}
// Workgroups take the positions u = 0, 1, 2, ... in turn, and workgroup b runs
// on XCD b % 8, so a position's XCD is u mod 8.  Each 8 chunk positions take as
// many consecutive windows, eight chunks that go one to each XCD.  Boxes of equal
// sides in a row repeat the same work every few windows (the first and the last
// of a box hold little of the band), so the eight chunks are rotated by a
// golden-ratio hash of their group.  A bijection on every multiple of 8 chunk.
constexpr int run_window(int u, int chunk) {
  const uint32_t group = (uint32_t)u / (8u * chunk), r = (uint32_t)u % (8u * chunk);
  const uint32_t turn = group * 2654435769u >> 29;
  return (int)(group * (8u * chunk) + ((r + turn) & 7u) * chunk + (r >> 3));
}
}  // namespace gg
