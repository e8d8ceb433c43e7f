// Layout rules shared by kernels and host code: plain C++ without device types,
// so that a host program can check them over their whole range.
#pragma once

namespace oal {

constexpr int kMore = 3;  // further windows of a head: 64 dimensions hold at most three beyond each group's first 16

// A window of 16 LDS positions that holds dimensions of one group. An absent one
// (group -1) is a valid empty window, since the token-pair kernels read every
// slot and drop what no group claims.
struct Window {
  int group = -1, at = 0, count = 0;
};

// Positions of the token-pair kernels' sorted rows (Lay in oal_direct.hip): groups
// 0, 1, .. of n dimensions each are passed in order.
template <bool F32, int GP>
struct WindowWalk {
  // the last window may start at the end
  static constexpr int kPositions = F32 ? 16 * (GP + kMore) : 64 + 3 * (GP - 1) + 16;
  int start = 0, more = 0;  // bf16: the group's first position; further windows so far

  constexpr int first(int g) const { return F32 ? 16 * g : start; }
  constexpr int next() const { return F32 ? 16 * (GP + more) : start + 16; }
  // A group of n dimensions has extra(n) further windows; number i of them goes into slot more + i.
  static constexpr int extra(int n) { return n > 16 ? (n + 15) / 16 - 1 : 0; }
  constexpr Window further(int i, int g, int n) const {
    const int left = n - 16 * (i + 1);
    return Window{g, next() + 16 * i, left < 16 ? left : 16};
  }
  constexpr void pass(int n) {
    more += extra(n);
    start += (n + 3) & ~3;
  }
};

// Grid of kernels with one block for each of `heads` (at most 65535) and each of
// `tiles`, the heads side by side: heads in x, tiles over y and, past its limit,
// z. (In x alone, tiles * heads blocks of 512 threads pass the 2^32 threads that a
// launch may have in one dimension.) Blocks with tile >= tiles have no work.
struct TileGrid {
  unsigned x, y, z;
};
constexpr unsigned kGridLimit = 65535;
constexpr TileGrid tile_grid(unsigned heads, unsigned tiles) {
  const unsigned z = (tiles + kGridLimit - 1) / kGridLimit;
  return {heads, (tiles + z - 1) / z, z};
}
constexpr unsigned tile_of(unsigned block_y, unsigned block_z, unsigned grid_y) { return block_z * grid_y + block_y; }

}  // namespace oal
