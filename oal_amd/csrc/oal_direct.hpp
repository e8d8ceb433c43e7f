// The direct route: evaluation over token pairs for short sequences
// (oal_direct.hip).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "oal_internal.hpp"

namespace oal {

constexpr int kDirectTile = 16;  // tokens per tile edge

// Whether a call takes the direct route: where a model of both routes' forward
// and backward time on MI355X (microseconds, kernels alone) says that it is the
// shorter one. A function of the geometry alone, so that the size queries and
// both directions agree. A direct call costs its launches and the longest row,
// its 16 x 16 tiles and its blocks of 16 rows; the state route its longer chain
// of launches (in bf16 with 30 us for what the host takes longer over them) and
// its rows. Measured, bf16, 14/2 heads and 8 groups, direct against state: B=1
// N=128 46 / 216, N=512 90 / 238, N=1024 177 / 257, N=1300 233 / 266, N=1600 299 /
// 277; B=2 N=800 196 / 274, N=1000 272 / 270, N=1200 335 / 315; B=8 N=512 394 /
// 315; B=64 N=128 404 / 437, N=256 1011 / 929. fp32: B=1 N=256 93 / 438, N=1024
// 426 / 586, N=1536 766 / 663; B=4 N=512 502 / 800, N=1024 1394 / 1202; B=64 N=256
// 2589 / 3814. Up to 4 groups: bf16 B=1 N=1600 228 / 280, B=4 N=1024 408 / 321;
// fp32 B=1 N=2048 629 / 769, B=4 N=1024 755 / 1171.
// All measured with the blocks numbered head by head. Longest rows of all heads
// first, a forward and backward take up to a quarter less (bf16 B=1 N=1024 160 to
// 130, B=2 N=1000 256 to 219, B=16 N=256 246 to 202; fp32 B=1 N=1024 382 to 274; no
// size slower), so the line is on the safe side for the direct route.
inline bool direct_route(bool f32, int groups, int B, int Hq, int N) {
  if (groups > 8 || (long)B * Hq > 65535) return false;
  const double nt = (N + kDirectTile - 1) / kDirectTile, blocks = (double)B * Hq * nt, tiles = blocks * (nt + 1) / 2,
               rows = (double)B * Hq * N;
  const bool few = groups <= 4;
  // One or two heads: the time is the longest row's chain, 61 ns a token and direction
  // (50 up to 4 groups) against the state's 21, which the terms below do not hold. One
  // head, 8 groups: N=3000 197 / 232, N=3600 237 / 245, N=3900 253 / 249, N=4390 285 /
  // 262; without gradients of the coefficients N=4416 273 / 248; two heads of one
  // unit N=3392 239 / 234. Up to 4 groups: N=4400 231 / 261, N=5000 270 / 277, without
  // coefficients N=5088 266 / 260.
  if (!f32 && N > (few ? 4500 : 3200)) return false;
  if (f32) return 60 + 0.03 * N + (few ? 0.0042 : 0.0082) * tiles + (few ? 0.06 : 0.085) * blocks < 420 + 0.0145 * rows;
  return 35 + 0.02 * N + (few ? 0.0018 : 0.0027) * tiles + (few ? 0.05 : 0.055) * blocks < 230 + 0.0028 * rows;
}

// Workspace of a direct backward.
size_t direct_work_bytes(bool f32, int B, int Hq, int N);

// F32: fp32 arithmetic, else bf16 operands with fp32 accumulation.
template <typename T, bool F32>
void launch_direct_forward(const LaunchGeom& g, const T* q, const T* k, const T* v, const int32_t* labels,
                           const float* c0, const float* lam, const float* gam, int groups, float scale, float floor,
                           T* out, float* num, float* den, hipStream_t st, const Timer& timed);
template <typename T, bool F32>
void launch_direct_backward(const LaunchGeom& g, const T* q, const T* k, const T* v, const int32_t* labels,
                            const float* c0, const float* lam, const float* gam, int groups, float scale, float floor,
                            const float* num, const float* den, const T* dout, const float* dnum, const float* dden,
                            T* dq, T* dk, T* dv, float* dc0, float* dlam, float* dgam, void* workspace, hipStream_t st,
                            const Timer& timed);

}  // namespace oal
