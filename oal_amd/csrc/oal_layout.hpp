// Layout rules shared by kernels and host code: plain C++ without device types,
// so that a host program can check them over their whole range.
#pragma once

namespace oal {

constexpr int kMore = 3;  // further windows of a head: 64 dimensions hold at most three beyond each group's first 16

// A further window packed into a word: its group, first position and count of
// dimensions. An absent one is group 255, an empty window at position 0.
struct Window {
  unsigned word = 255u << 16;
  constexpr int group() const { return (int)(word >> 16); }
  constexpr int at() const { return (int)(word >> 8 & 255u); }
  constexpr int count() const { return (int)(word & 255u); }
  constexpr bool present() const { return group() != 255; }
};

// Positions of the token-pair kernels' sorted rows (Lay in oal_direct.hip): groups
// 0, 1, .. of n dimensions each are passed in order.
template <bool F32, int GP>
struct WindowWalk {
  // the last window may start at the end
  static constexpr int kPositions = F32 ? 16 * (GP + kMore) : 64 + 3 * (GP - 1) + 16;
  static_assert(kPositions <= 256, "a position fits a byte");
  int start = 0, more = 0;  // bf16: the group's first position; further windows so far

  constexpr int first(int g) const { return F32 ? 16 * g : start; }
  constexpr int next() const { return F32 ? 16 * (GP + more) : start + 16; }
  // Passes group g of n dimensions; its further windows go into the next slots.
  constexpr void pass(int g, int n, Window (&slot)[kMore]) {
    if (n > 16) {
      const int extra = (n + 15) / 16 - 1;
      for (int m = 0; m < kMore; ++m) {
        const int i = m - more, left = n - 16 * (i + 1);
        if (i >= 0 && i < extra)
          slot[m].word = (unsigned)g << 16 | (unsigned)(next() + 16 * i) << 8 | (unsigned)(left < 16 ? left : 16);
      }
      more += extra;
    }
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
