// The direct route: evaluation over token pairs for short sequences
// (oal_direct.hip).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "oal_internal.hpp"

namespace oal {

constexpr int kDirectTile = 16;  // tokens per tile edge

// Whether a call takes the direct route: where a model of both routes' forward
// and backward time on MI355X (microseconds of the library's calls in turn) says
// that it is the shorter one. A function of the geometry alone, so that the size
// queries and both directions agree. A direct call costs its launches and the longest
// row, its 16 x 16 tiles and its blocks of 16 rows; the state route its longer
// chain of launches (in bf16 with 30 us for what the host takes longer over them)
// and its rows. Measured forward and backward, direct against state, at 14/2 heads
// and, last of each list, at the line:
//   bf16, 8 groups   B=1 N=712 84 / 239, N=1139 155 / 254, N=1424 207 / 262; B=2 N=1008
//                    212 / 254; B=4 N=704 225 / 283; B=16 N=336 305 / 404; B=64 N=144 412 / 560
//   bf16, 4 groups   B=1 N=848 82 / 246, N=1356 158 / 257, N=1696 205 / 265; B=16 N=416 301 / 475
//   fp32, 8 groups   B=1 N=744 192 / 506, N=1190 349 / 617, N=1488 472 / 640; B=4 N=944
//                    804 / 1098; B=16 N=688 1915 / 2664; B=64 N=592 6083 / 8994
//   fp32, 4 groups   B=1 N=1144 201 / 548, N=1830 398 / 694, N=2288 568 / 791; B=16 N=1344 3437 / 4580
// The host does not see the labels, so the line also holds for heads whose groups are
// long (sizes 57 and seven of 1: bf16 B=1 N=1424 253 / 258, fp32 B=16 N=688 2377 / 2781;
// 61, 1, 1, 1: bf16 B=1 N=1696 239 / 265, fp32 B=16 N=1344 4720 / 4679). For even groups it
// is on the safe side. It does not know the number of KV heads, which the state's scans
// run over (measured with 1 to 32, none slower), nor 64-token chunks: many
// sequences of a few tokens, and calls without a backward, take its line as it is.
inline bool direct_route(bool f32, int groups, int B, int Hq, int N) {
  if (groups > 8 || (long)B * Hq > 65535) return false;
  const double nt = (N + kDirectTile - 1) / kDirectTile, blocks = (double)B * Hq * nt, tiles = blocks * (nt + 1) / 2,
               rows = (double)B * Hq * N;
  const bool few = groups <= 4;
  // Fewer than four groups hold one of more than 16 dimensions, whose further windows cost more.
  const double tile = f32 ? (groups > 4 ? 0.0082 : groups == 4 ? 0.0044 : 0.0048)
                          : (groups > 4 ? 0.0027 : groups == 4 ? 0.0019 : 0.0021);
  // One or two heads in bf16: the time is the longest row's chain, which the terms
  // below do not hold, 61 to 82 ns a token with 8 groups against the state's 20. One
  // head, even groups: N=3000 197 / 232, N=3900 253 / 249, N=4390 285 / 262; sizes 57
  // and seven of 1: N=2400 218 / 221, N=3200 284 / 236. Four groups: N=4199 even 232 /
  // 261, sizes 61, 1, 1, 1 N=3149 223 / 238, N=4199 291 / 259.
  if (!f32 && N > (few ? 3200 : 2400)) return false;
  if (f32) return 60 + 0.03 * N + tile * tiles + (few ? 0.06 : 0.085) * blocks < 420 + 0.0145 * rows;
  return 35 + 0.02 * N + tile * tiles + (few ? 0.05 : 0.055) * blocks < 230 + 0.0028 * rows;
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
