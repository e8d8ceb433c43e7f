"""Rules of oal_amd/csrc/oal_layout.hpp over their whole range, in a host program:
what the kernels read by them stays inside its arrays."""

import os
import shutil
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "oal_amd", "csrc")


def _run(tmp_path, source):
    cxx = shutil.which("g++") or shutil.which("c++")
    if cxx is None:
        pytest.skip("no host C++ compiler")
    src, exe = tmp_path / "rule.cpp", tmp_path / "rule"
    src.write_text(source)
    subprocess.run([cxx, "-std=c++20", "-O1", "-Wall", "-Werror", "-I" + CSRC, str(src), "-o", str(exe)], check=True)
    done = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert done.returncode == 0, done.stdout


def test_every_window_slot_is_inside_the_sorted_row(tmp_path):
    """The token-pair kernels read further windows at LDS positions: every slot, present
    or not, is an aligned window inside the row, and the windows hold all 64
    dimensions. Every size of up to three groups, and random sizes of all."""
    _run(tmp_path, r"""
#include <cstdio>
#include <cstdlib>
#include <random>
#include <vector>
#include "oal_layout.hpp"
using namespace oal;

template <bool F32, int GP>
void check(const std::vector<int>& sizes) {
  using Walk = WindowWalk<F32, GP>;
  Window table[kMore];
  int held = 0;
  Walk walk;
  for (int g = 0; g < GP; ++g) {
    const int n = g < (int)sizes.size() ? sizes[g] : 0, before = walk.more;
    if (walk.first(g) % 4 || walk.first(g) < 0 || walk.first(g) + 16 > Walk::kPositions) std::exit(1);
    held += n < 16 ? n : 16;
    walk.pass(g, n, table);
    if (walk.more > kMore || walk.more - before != (n > 16 ? (n + 15) / 16 - 1 : 0)) std::exit(2);
  }
  for (int x = 0; x < kMore; ++x) {
    const Window& w = table[x];
    const bool ok = w.at() >= 0 && w.at() % 4 == 0 && w.at() + 16 <= Walk::kPositions && w.present() == (x < walk.more) &&
                    (w.present() ? w.group() < GP && w.count() > 0 && w.count() <= 16 : w.count() == 0 && w.at() == 0);
    if (!ok) {
      std::printf("F32=%d GP=%d: window %d %d %d\n", F32, GP, w.group(), w.at(), w.count());
      std::exit(3);
    }
    held += w.count();
  }
  if (held != 64) std::exit(4);
}
void all(const std::vector<int>& sizes) {
  if (sizes.size() <= 4) {
    check<false, 4>(sizes);
    check<true, 4>(sizes);
  }
  check<false, 8>(sizes);
  check<true, 8>(sizes);
}
int main() {
  for (int a = 0; a <= 64; ++a)
    for (int b = 0; a + b <= 64; ++b) all({a, b, 64 - a - b});
  std::mt19937 rng(1);
  for (int i = 0; i < 200000; ++i) {
    std::vector<int> sizes(1 + rng() % 8);
    const int few = 1 + rng() % sizes.size();
    for (int d = 0; d < 64; ++d) ++sizes[rng() % few * sizes.size() / few];
    all(sizes);
  }
}
""")


def test_the_float64_group_kernels_grid_stays_inside_the_launch_limits(tmp_path):
    """Every (batch, head) and sequence length that the float64 entry points take
    (65535 heads, 65535 32-token tiles): each tile has one block, y and z stay under
    65536, and no dimension reaches 2^32 threads of 512-thread blocks."""
    _run(tmp_path, r"""
#include <initializer_list>
#include "oal_layout.hpp"
using namespace oal;
int main() {
  for (unsigned heads : {1u, 14u, 4096u, 65535u})
    for (unsigned tiles = 1; tiles <= 131070; tiles = tiles < 3000 ? tiles + 1 : tiles + 7) {
      const TileGrid g = tile_grid(heads, tiles);
      if (g.x * 512ull >= 1ull << 32 || g.x != heads || g.y > 65535 || g.z > 65535) return 1;
      const unsigned last = tile_of(g.y - 1, g.z - 1, g.y);
      if (last < tiles - 1 || tile_of(0, g.z - 1, g.y) >= tiles || tile_of(0, 1, g.y) != g.y) return 2;
    }
  const TileGrid g = tile_grid(65535, 131070);
  return g.y * g.z < 131070;
}
""")
