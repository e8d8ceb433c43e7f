// Direct evaluation over token pairs for gfx950, up to 8 groups: the route of
// sequences short enough that O(N^2) pairs cost less than the O(N) running
// state over 2145 features (direct_route in oal_direct.hpp has the line and
// both sides of it).
//
//   s_g(i,j) = sum_{d in g} q_i[d] k_j[d],  kappa = c0 + sum_g s_g (a_g + sum_h A_gh s_h)
//   a_g = scale lam_g,  A_gh = scale^2 gam_gh
//   num_i = sum_{j<=i} kappa v_j,  den_i = sum_{j<=i} kappa,  out_i = num_i / max(den_i, floor)
// and the VJP with G, Gz from the normalization (k2_bwd_prep's formulas):
//   ds = G_i . v_j + Gz_i,  t_g = a_g + 2 sum_h A_gh s_h
//   dq_i[d] = sum_j ds t_g(d) k_j[d],  dk_j[d] = sum_i ds t_g(d) q_i[d],  dv_j = sum_i kappa G_i
//   dc0 = sum ds,  dlam_g = scale sum ds s_g,  dgam_gh = scale^2 sum ds s_g s_h
// (reference grouped_reference.py:102-211 over pairs; backward as in
// oal_mfma_local.hip, whose chunk becomes the whole sequence).
//
// Nothing but q, k, v, num and den is read back by the backward: no state is
// saved and the workspace holds G and the per-head dk, dv.
//
// A block owns 16 rows of the fixed side and streams 16-row tiles of the other:
//   forward  fixed q          streamed k, v   num, den, out
//   dq       fixed q, G       streamed k, v   dq, coefficient sums; also forms G
//   dkv      fixed k, v       streamed q, G   dk, dv of one query head
// Per 16 x 16 tile the group sums come from the matrix cores, the quadratic form
// is VALU work in fp32 and the tile goes back into the matrix cores as it stands
// in the accumulator layout: entry [4 (l / 16) + r][l % 16], which is the first
// operand of a product over the streamed rows. In direct_tiles (the forward, and
// the fp32 backward) the four waves take tiles in turn and add up in wave order at
// the end; a tile costs a lane 44 FMAs for kappa, in the backward 64 for the
// slopes and 45 for the coefficient sums, times four entries: VALU issue bounds
// it in bf16, matrix-core issue in fp32 (v_mfma_f32_16x16x4_f32: 32 cycles for a
// sixteenth of the bf16 depth). The bf16 backward is in direct_dq and
// direct_dk_dv (roles). In short sequences what counts is the chain from the first
// load to the first tile, so every wave works its group structure out for itself
// without a barrier; N = 64, 14 heads, takes 7 us forward and 31 forward and
// backward, against 44 and 197 through the state. At full load the waves' VALU and
// matrix-core cycles add up to the time (they hardly overlap): a step of 64 rows of
// the bf16 dq is about 360 VALU and 52 matrix instructions a wave.
//
// The dimensions are sorted by group in LDS, a window of 16 positions for each
// group's first 16 dimensions and at most three more in all. A group's sum is then
// one product over its own window instead of a masked product over all 64
// dimensions (and, in fp32, its gradient product fills its own columns).

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "oal_direct.hpp"
#include "oal_internal.hpp"
#include "oal_layout.hpp"
#include "oal_mfma_common.hpp"

namespace oal {

namespace {

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

constexpr int kM = kDirectTile;  // tile edge
constexpr int kWv = 4;           // waves per block

enum Mode { kFwd, kDq, kDkv, kDk, kDv };

constexpr int kStep = kM * kWv;  // streamed rows that a block's waves share (bf16 backward)

// Coefficient sums of a tile: sum ds {1, s_g, s_g s_h (h <= g)}, or sum ds and sum ds s_h s_g for all (h, g), s_GP = 1.
constexpr int coef_count(int gp) { return 1 + gp + gp * (gp + 1) / 2; }
constexpr int role_coef_count(int gp) { return 1 + (gp + 1) * gp; }

__device__ __forceinline__ void store4(float* dst, const float4& y) { *reinterpret_cast<float4*>(dst) = y; }
__device__ __forceinline__ void store4(uint16_t* dst, const float4& y) {
  *reinterpret_cast<uint2*>(dst) = make_uint2(pack_bf16x2(y.x, y.y), pack_bf16x2(y.z, y.w));
}

// Element type of the staged tiles and of G: bf16, or fp32 for the fp32 arithmetic.
template <bool F32>
using Elem = std::conditional_t<F32, float, uint16_t>;

// 16 consecutive elements of a row: dimensions 16 (l % 4) .. of row l / 4.
template <typename T>
struct Piece;
template <>
struct Piece<uint16_t> {
  u32x4 w[2];
};
template <>
struct Piece<float> {
  float4 f[4];
};
__device__ __forceinline__ void load_piece(Piece<uint16_t>& p, const uint16_t* src) {
  p.w[0] = reinterpret_cast<const u32x4*>(src)[0];
  p.w[1] = reinterpret_cast<const u32x4*>(src)[1];
}
__device__ __forceinline__ void load_piece(Piece<float>& p, const float* src) {
#pragma unroll
  for (int x = 0; x < 4; ++x) p.f[x] = reinterpret_cast<const float4*>(src)[x];
}
__device__ __forceinline__ float4 piece4(const Piece<float>& p, int x) { return p.f[x]; }
__device__ __forceinline__ float4 piece4(const Piece<uint16_t>& p, int x) {
  const uint32_t a = p.w[x >> 1][2 * (x & 1)], b = p.w[x >> 1][2 * (x & 1) + 1];
  return make_float4(__uint_as_float(a << 16), __uint_as_float(a & 0xffff0000u), __uint_as_float(b << 16),
                     __uint_as_float(b & 0xffff0000u));
}
__device__ __forceinline__ uint32_t piece_word(const Piece<uint16_t>& p, int x) { return p.w[x >> 2][x & 3]; }
__device__ __forceinline__ uint32_t piece_word(const Piece<float>& p, int x) {
  const float4 f = p.f[x >> 1];
  return x & 1 ? pack_bf16x2(f.z, f.w) : pack_bf16x2(f.x, f.y);
}
// Row of the streamed or fixed tile that this lane's piece belongs to; rows
// past N repeat the last one (their pairs are masked).
template <typename T>
__device__ __forceinline__ void load_tile(Piece<T>& p, const T* __restrict__ base, int row0, int N, int l) {
  const int row = row0 + (l >> 2);
  load_piece(p, base + (size_t)(row < N ? row : N - 1) * kD + 16 * (l & 3));
}

// LDS layout of a tile's rows.
//   natural  [64]
//   sorted   windows of 16 positions, one for each group's first 16 dimensions and
//            up to kMore for the rest. bf16: a group starts at a multiple of four
//            positions and its windows follow it, overlapping the next group
//            (the fixed operand is zero there). fp32: every window is a block of
//            its own, position p at 4 (p % 4) + p / 4, so that the four k-steps of
//            lane group p % 4 are one 16-byte read.
template <bool F32, int GP>
struct Lay {
  static constexpr int kWin = GP + kMore;
  static constexpr int kPos = WindowWalk<F32, GP>::kPositions;
  static constexpr int LS = F32 ? kPos + 4 : (kPos + 7) / 8 * 8 + 4;
  static constexpr int LN = kD + (F32 ? 4 : 8);
  static __device__ __forceinline__ constexpr int in_block(int p) { return F32 ? 4 * (p & 3) + (p >> 2) : p; }
};

template <bool F32, int GP>
struct Shared {
  using L = Lay<F32, GP>;
  Elem<F32> sorted[kWv][kM][L::LS];
  Elem<F32> natural[kWv][kM][L::LN];
  Elem<F32> fixed[kM][L::LS];
  uint8_t dim[16 * L::kWin];  // fp32: window and position -> dimension, 255 where there is none
  uint32_t more[kMore];  // further windows (Window::word)
  float zrow[kWv][kM];
  float co[kWv][coef_count(GP)];
};

// A head's labels and coefficients, held across a wave's lanes, and its group
// structure in scalar registers: every wave works them out for itself from one
// load each, with no table in memory and no barrier.
template <bool F32, int GP>
struct Head {
  int lab;           // lane = dimension: its group
  int pos;           // its LDS position
  float gam, lam;    // lane 8 g + h: scale^2 gam[g][h]; lane g: scale lam[g]
  int at[GP], count[GP];  // a group's first window and its dimensions in it
  bool any_more;          // whether there are further windows (groups of more than 16 dimensions)
};

template <bool F32, int GP>
__device__ __forceinline__ Head<F32, GP> read_head(const int32_t* __restrict__ labels, const float* __restrict__ lam,
                                                   const float* __restrict__ gam, int G, int h, float scale, int l,
                                                   uint32_t (&more)[kMore]) {
  using L = Lay<F32, GP>;
  Head<F32, GP> t;
  const int x = l >> 3, y = l & 7;
  const float gv = gam[((size_t)h * G + min(x, G - 1)) * G + min(y, G - 1)], lv = lam[(size_t)h * G + min(l, G - 1)];
  const int own = labels[h * kD + l];
  t.lab = own < 0 ? 0 : (own >= G ? G - 1 : own);
  t.gam = x < G && y < G ? scale * scale * gv : 0.f;
  t.lam = l < G ? scale * lv : 0.f;
  WindowWalk<F32, GP> walk;
  Window slot[kMore];
  t.pos = 0;
#pragma unroll
  for (int g = 0; g < GP; ++g) {
    const uint64_t in = __ballot(t.lab == g);
    const int n = __popcll(in);
    t.at[g] = walk.first(g);
    t.count[g] = min(16, n);
    const int i = __builtin_amdgcn_mbcnt_hi((uint32_t)(in >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)in, 0));
    const int w = i < 16 ? t.at[g] : walk.next() + (i & ~15) - 16;
    t.pos = t.lab == g ? w + L::in_block(i & 15) : t.pos;
    walk.pass(g, n, slot);
  }
  // in LDS, since few heads have any and in scalar registers they displace the coefficients
  if (threadIdx.x < kMore)
    more[threadIdx.x] = threadIdx.x == 0 ? slot[0].word : threadIdx.x == 1 ? slot[1].word : slot[2].word;
  t.any_more = walk.more > 0;
  return t;
}

// Byte offsets of this lane's 16 elements (dimensions 16 (l % 4) ..) in the sorted
// tile of 16 rows that starts at row row0 of an array: added to the array's own
// (constant) LDS address they cost a write no instruction.
template <bool F32, int GP>
__device__ __forceinline__ void piece_offsets(int (&off)[16], const Head<F32, GP>& t, int row0, int l) {
#pragma unroll
  for (int e = 0; e < 16; ++e)
    off[e] = (int)sizeof(Elem<F32>) * ((row0 + (l >> 2)) * Lay<F32, GP>::LS + __shfl(t.pos, 16 * (l & 3) + e, 64));
}
template <typename E>
__device__ __forceinline__ E& at_byte(E* p, int off) {
  return *reinterpret_cast<E*>(reinterpret_cast<char*>(p) + off);
}

template <typename T>
__device__ __forceinline__ void put_sorted(uint16_t* tile, const Piece<T>& p, const int (&off)[16]) {
#pragma unroll
  for (int x = 0; x < 8; ++x) {
    const uint32_t w = piece_word(p, x);
    at_byte(tile, off[2 * x]) = (uint16_t)w;
    at_byte(tile, off[2 * x + 1]) = (uint16_t)(w >> 16);
  }
}
template <typename T>
__device__ __forceinline__ void put_sorted(float* tile, const Piece<T>& p, const int (&off)[16]) {
#pragma unroll
  for (int x = 0; x < 4; ++x) {
    const float4 f = piece4(p, x);
    at_byte(tile, off[4 * x]) = f.x;
    at_byte(tile, off[4 * x + 1]) = f.y;
    at_byte(tile, off[4 * x + 2]) = f.z;
    at_byte(tile, off[4 * x + 3]) = f.w;
  }
}
template <int LN, typename T>
__device__ __forceinline__ void put_natural(uint16_t* tile, const Piece<T>& p, int l) {
  u32x4* dst = reinterpret_cast<u32x4*>(tile + (l >> 2) * LN + 16 * (l & 3));
#pragma unroll
  for (int x = 0; x < 2; ++x)
    dst[x] = u32x4{piece_word(p, 4 * x), piece_word(p, 4 * x + 1), piece_word(p, 4 * x + 2), piece_word(p, 4 * x + 3)};
}
template <int LN, typename T>
__device__ __forceinline__ void put_natural(float* tile, const Piece<T>& p, int l) {
  float4* dst = reinterpret_cast<float4*>(tile + (l >> 2) * LN + 16 * (l & 3));
#pragma unroll
  for (int x = 0; x < 4; ++x) dst[x] = piece4(p, x);
}

// Orders a wave's LDS writes before its lanes' reads of one another's (a wave's
// LDS operations complete in order; this keeps the compiler from moving them).
__device__ __forceinline__ void wave_order() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// One window of 16 positions: first operand (row l % 16), second operand (column
// l % 16), and the product over the 16 positions.
template <bool F32>
struct Blk;
template <>
struct Blk<false> {
  s16x4 v;
};
template <>
struct Blk<true> {
  f32x4 v;
};
template <bool F32>
__device__ __forceinline__ Blk<F32> read_window(const Elem<F32>* row, int at, int l) {
  Blk<F32> b;
  b.v = *reinterpret_cast<const decltype(b.v)*>(row + at + 4 * (l >> 4));
  return b;
}
// The same at a lane's precomputed offset in a sorted tile (window_offset), one
// register a window instead of an addition a read.
template <bool F32, int GP>
__device__ __forceinline__ int window_offset(int at, int l) {
  return (l & 15) * Lay<F32, GP>::LS + at + 4 * (l >> 4);
}
template <bool F32>
__device__ __forceinline__ Blk<F32> read_at(const Elem<F32>* tile, int offset) {
  Blk<F32> b;
  b.v = *reinterpret_cast<const decltype(b.v)*>(tile + offset);
  return b;
}
__device__ __forceinline__ Window more_window(const uint32_t (&more)[kMore], int m) {
  Window w;
  w.word = __builtin_amdgcn_readfirstlane(more[m]);
  return w;
}
// The fixed operand of a window: zero past the group's own dimensions.
__device__ __forceinline__ Blk<false> fixed_window(const uint16_t* row, int at, int count, int l) {
  Blk<false> b = read_window<false>(row, at, l);
#pragma unroll
  for (int j = 0; j < 4; ++j) b.v[j] = 4 * (l >> 4) + j < count ? b.v[j] : (short)0;
  return b;
}
__device__ __forceinline__ Blk<true> fixed_window(const float* row, int at, int, int l) {
  return read_window<true>(row, at, l);
}
__device__ __forceinline__ f32x4 mma(const Blk<false>& a, const Blk<false>& b, f32x4 c) {
  return mfma16k16(a.v, b.v, c);
}
__device__ __forceinline__ f32x4 mma(const Blk<true>& a, const Blk<true>& b, f32x4 c) {
#pragma unroll
  for (int s = 0; s < 4; ++s) c = __builtin_amdgcn_mfma_f32_16x16x4f32(a.v[s], b.v[s], c, 0, 0, 0);
  return c;
}

// Second operand of a product over the tile's rows: columns col0 + 0 .. 15 of the
// rows 4 (l / 16) + 0 .. 3 of an LDS tile (col: the lane's own column in fp32).
__device__ __forceinline__ Blk<false> rows_operand(const uint16_t* tile, int LD, int col0, int, int l) {
  const int i = l & 15;
  typedef __attribute__((address_space(3))) trv4 lds_trv4;
  const uint16_t* p = tile + (4 * (l >> 4) + (i >> 2)) * LD + col0 + 4 * (i & 3);
  Blk<false> b;
  b.v = __builtin_bit_cast(s16x4, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_trv4*)(p)));
  return b;
}
__device__ __forceinline__ Blk<true> rows_operand(const float* tile, int LD, int col0, int col, int l) {
  const float* p = tile + 4 * (l >> 4) * LD + col0 + col;
  Blk<true> b;
#pragma unroll
  for (int r = 0; r < 4; ++r) b.v[r] = p[r * LD];
  return b;
}
template <bool F32>
__device__ __forceinline__ Blk<F32> as_operand(const f32x4& x) {
  Blk<F32> b;
  if constexpr (F32) {
    b.v = x;
  } else {
    const float y[4] = {x[0], x[1], x[2], x[3]};
    b.v = pack4(y);
  }
  return b;
}

// x as a sum of bf16 parts, each what the ones before leave: x to 2^-9, 2^-17 or
// (24 bits) 2^-25 with one, two or three.
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
template <int PARTS>
__device__ __forceinline__ void split4(s16x4 (&h)[PARTS], const float (&x)[4]) {
  float y[4] = {x[0], x[1], x[2], x[3]};
#pragma unroll
  for (int p = 0; p < PARTS; ++p) {
    const u32x2 w = {pack_bf16x2(y[0], y[1]), pack_bf16x2(y[2], y[3])};
#pragma unroll
    for (int r = 0; r < 4; ++r)
      y[r] -= __uint_as_float(r & 1 ? w[r >> 1] & 0xffff0000u : w[r >> 1] << 16);
    h[p] = __builtin_bit_cast(s16x4, w);
  }
}

// The whole 64-wide row as operand (ds = G . v): bf16 two 32-wide k-steps, fp32
// sixteen, step s of lane group g being position 16 g + s.
template <bool F32>
struct Row;
template <>
struct Row<false> {
  bf16x8 v[2];
};
template <>
struct Row<true> {
  f32x4 v[4];
};
template <int LN>
__device__ __forceinline__ Row<false> read_row(const uint16_t* tile, int l) {
  Row<false> r;
#pragma unroll
  for (int ks = 0; ks < 2; ++ks)
    r.v[ks] = *reinterpret_cast<const bf16x8*>(tile + (l & 15) * LN + 32 * ks + 8 * (l >> 4));
  return r;
}
template <int LN>
__device__ __forceinline__ Row<true> read_row(const float* tile, int l) {
  Row<true> r;
#pragma unroll
  for (int x = 0; x < 4; ++x)
    r.v[x] = *reinterpret_cast<const f32x4*>(tile + (l & 15) * LN + 16 * (l >> 4) + 4 * x);
  return r;
}
__device__ __forceinline__ f32x4 mma(const Row<false>& a, const Row<false>& b, f32x4 c) {
#pragma unroll
  for (int ks = 0; ks < 2; ++ks) c = mfma16(a.v[ks], b.v[ks], c);
  return c;
}
__device__ __forceinline__ f32x4 mma(const Row<true>& a, const Row<true>& b, f32x4 c) {
#pragma unroll
  for (int s = 0; s < 16; ++s) c = __builtin_amdgcn_mfma_f32_16x16x4f32(a.v[s >> 2][s & 3], b.v[s >> 2][s & 3], c, 0, 0, 0);
  return c;
}

// A head's scaled coefficients in scalar registers (zero beyond G groups):
// quad[g (g + 1) / 2 + h] = 2 A_gh for h < g; the diagonal is A_gg for kappa
// alone, 2 A_gg where the slopes are formed (kappa then follows from them).
template <int GP>
struct Coef {
  float c0, lin[GP], quad[GP * (GP + 1) / 2];
};
__device__ __forceinline__ float lane_value(float x, int lane) {
  return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(x), lane));
}
template <bool SLOPES, bool F32, int GP>
__device__ __forceinline__ Coef<GP> head_coefficients(const Head<F32, GP>& t, float c0, int l) {
  const float twice = 2.f * t.gam, held = !SLOPES && l % 9 == 0 ? t.gam : twice;  // lanes 8 g + g
  Coef<GP> c;
  c.c0 = c0;
#pragma unroll
  for (int g = 0; g < GP; ++g) {
    c.lin[g] = lane_value(t.lam, g);
#pragma unroll
    for (int x = 0; x <= g; ++x) c.quad[g * (g + 1) / 2 + x] = lane_value(held, 8 * g + x);
  }
  return c;
}
template <int GP>
__device__ __forceinline__ float quad_of(const Coef<GP>& c, int g, int h) {
  return g >= h ? c.quad[g * (g + 1) / 2 + h] : c.quad[h * (h + 1) / 2 + g];
}

// kappa alone: c0 + sum_g s_g (a_g + A_gg s_g + sum_{h < g} 2 A_gh s_h)
template <int GP>
__device__ __forceinline__ float kappa_of(const Coef<GP>& c, const f32x4 (&s)[GP], int r) {
  float k = c.c0;
#pragma unroll
  for (int g = 0; g < GP; ++g) {
    float t = c.lin[g];
#pragma unroll
    for (int h = 0; h <= g; ++h) t = fmaf(quad_of(c, g, h), s[h][r], t);
    k = fmaf(s[g][r], t, k);
  }
  return k;
}
// d kappa / d s_g = a_g + sum_h 2 A_gh s_h
template <int GP>
__device__ __forceinline__ float slope(const Coef<GP>& c, const f32x4 (&s)[GP], int g, int r) {
  float t = c.lin[g];
#pragma unroll
  for (int h = 0; h < GP; ++h) t = fmaf(quad_of(c, g, h), s[h][r], t);
  return t;
}

template <typename T, bool F32>
struct Args {
  const T *q, *k, *v;
  const int32_t* labels;
  const float *c0, *lam, *gam;
  int G, Hq, Hkv, N;
  float scale, floor;
  // forward
  T* out;
  float *num, *den;
  // backward
  const T* dout;
  const float *dnum, *dden;
  Elem<F32>* Gv;  // [B][Hq][N][64]
  float* Gz;      // [B][Hq][N]
  T* dq;          // nullptr: not requested
  float* part;    // [B * Hq][tiles][coef_count] coefficient sums, nullptr: not requested
  float *dkh, *dvh;  // [B][Hq][N][64] per query head
};

// The rows' G and Gz for the block's 16 query rows (k2_bwd_prep's formulas):
// every wave forms them for itself, wave 0 writes them out for the dkv kernel.
template <typename T, bool F32>
__device__ __forceinline__ void normalization_vjp(Piece<Elem<F32>>& gp, float& gz, const Args<T, F32>& a, int bh,
                                                  int row0, int wave, int l) {
  const int row = row0 + (l >> 2);
  const bool ok = row < a.N;
  const size_t at = (size_t)bh * a.N + (ok ? row : a.N - 1), o = at * kD + 16 * (l & 3);
  float g[16], dot = 0.f;
  const float dd = a.den[at];
  const float dp = a.floor > 0.f ? fmaxf(dd, a.floor) : dd, inv = 1.f / dp;
  // bf16: G is rounded to 8 bits, so the reciprocal's rounding does not count
  auto over = [&](float x) { return F32 ? x / dp : x * inv; };
#pragma unroll
  for (int e = 0; e < 16; ++e) g[e] = 0.f;
  if (a.dout) {
    Piece<T> x;
    Piece<float> nm;
    load_piece(x, a.dout + o);
    load_piece(nm, a.num + o);
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const float4 y = piece4(x, e), n = piece4(nm, e);
      dot = fmaf(y.x, n.x, fmaf(y.y, n.y, fmaf(y.z, n.z, fmaf(y.w, n.w, dot))));
      g[4 * e] = over(y.x);
      g[4 * e + 1] = over(y.y);
      g[4 * e + 2] = over(y.z);
      g[4 * e + 3] = over(y.w);
    }
  }
  if (a.dnum) {
    Piece<float> x;
    load_piece(x, a.dnum + o);
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const float4 y = piece4(x, e);
      g[4 * e] += y.x;
      g[4 * e + 1] += y.y;
      g[4 * e + 2] += y.z;
      g[4 * e + 3] += y.w;
    }
  }
  dot += __shfl_xor(dot, 1, 64);
  dot += __shfl_xor(dot, 2, 64);
  gz = -dot / (dp * dp);
  if (a.floor > 0.f && !(dd >= a.floor)) gz = 0.f;
  if (a.dden) gz += a.dden[at];
  if (!ok) {
    gz = 0.f;
#pragma unroll
    for (int e = 0; e < 16; ++e) g[e] = 0.f;
  }
  if constexpr (F32) {
#pragma unroll
    for (int x = 0; x < 4; ++x) gp.f[x] = make_float4(g[4 * x], g[4 * x + 1], g[4 * x + 2], g[4 * x + 3]);
  } else {
#pragma unroll
    for (int x = 0; x < 8; ++x) gp.w[x >> 2][x & 3] = pack_bf16x2(g[2 * x], g[2 * x + 1]);
  }
  if (wave == 0 && ok) {
    if constexpr (F32) {
#pragma unroll
      for (int x = 0; x < 4; ++x) reinterpret_cast<float4*>(a.Gv + o)[x] = gp.f[x];
    } else {
      reinterpret_cast<u32x4*>(a.Gv + o)[0] = gp.w[0];
      reinterpret_cast<u32x4*>(a.Gv + o)[1] = gp.w[1];
    }
    if ((l & 3) == 0) a.Gz[at] = gz;
  }
}

// Zeroes an LDS array (its size a multiple of 8 bytes), all threads of the block.
template <typename A>
__device__ __forceinline__ void zero_lds(A& x) {
  static_assert(sizeof(A) % 8 == 0, "whole 8-byte words");
  for (int i = threadIdx.x; i < (int)(sizeof(A) / 8); i += blockDim.x)
    reinterpret_cast<uint2*>(&x)[i] = make_uint2(0, 0);
}

// Adds the waves' column blocks into an LDS tile [16][64] in wave order:
// put(w) is called for wave w between two barriers, by that wave alone.
template <typename F>
__device__ __forceinline__ void in_wave_order(int wave, F&& put) {
#pragma unroll 1
  for (int w = 0; w < kWv; ++w) {
    if (w == wave) put(w == 0);
    __syncthreads();
  }
}

}  // namespace

template <typename T, bool F32, int GP, int MODE>
__device__ __forceinline__ void tiles(const Args<T, F32>& a, Shared<F32, GP>& sh) {
  constexpr bool kSums = MODE == kFwd || MODE == kDv;   // products with kappa alone
  constexpr bool kKeys = MODE == kDkv || MODE == kDv;   // the fixed rows are keys
  static_assert(kSums || F32, "the rest of the bf16 backward is in roles");
  using L = Lay<F32, GP>;
  using E = Elem<F32>;
  const int wave = threadIdx.x >> 6, l = threadIdx.x & 63, lr = l & 15, lg = l >> 4;
  const int NT = gridDim.y, bh = blockIdx.x, N = a.N;
  // the tiles with the most pairs first, of all heads: the last ones to start are
  // short (the rows of one head after another: forward at B=2, N=1000, 14 heads 51 us, not 41)
  const int ft = kKeys ? (int)blockIdx.y : NT - 1 - (int)blockIdx.y;
  const int R = a.Hq / a.Hkv, b = bh / a.Hq, h = bh % a.Hq, u = b * a.Hkv + h / R;
  const size_t qbase = (size_t)bh * N * kD, kbase = (size_t)u * N * kD;
  const int row0 = ft * kM;

  const float c0 = a.c0[h];
  const Head<F32, GP> hd = read_head<F32, GP>(a.labels, a.lam, a.gam, a.G, h, a.scale, l, sh.more);
  // zero the sorted tiles once: the padding positions stay zero
  zero_lds(sh.sorted);
  zero_lds(sh.fixed);
  if constexpr (!kSums) {
    for (int x = threadIdx.x; x < 16 * L::kWin; x += 64 * kWv) sh.dim[x] = 255;
  }
  int off[16];
  piece_offsets(off, hd, wave * kM, l);
  __syncthreads();
  if constexpr (!kSums) {
    // fp32 positions run 4 (p % 4) + p / 4 within a window
    if (wave == 0) sh.dim[(hd.pos & ~15) + ((hd.pos & 3) * 4 + ((hd.pos >> 2) & 3))] = (uint8_t)l;
  }
  const Coef<GP> cf = head_coefficients<!kSums>(hd, c0, l);

  E* const srt = &sh.sorted[wave][0][0];
  E* const nat = &sh.natural[wave][0][0];
  // fixed side: its sorted rows in LDS for the block, its natural rows (dq: G,
  // dkv: v) as each wave's operand
  Row<F32> f2{};
  float gzc = 0.f;  // dq: Gz of the lane's query column
  {
    Piece<T> p;
    load_tile(p, kKeys ? a.k + kbase : a.q + qbase, row0, N, l);
    if (wave == 0) put_sorted(&sh.fixed[0][0], p, off);
    if constexpr (MODE == kDq) {
      Piece<E> gp;
      float gz;
      normalization_vjp<T, F32>(gp, gz, a, bh, row0, wave, l);
      put_natural<L::LN>(nat, gp, l);
      gzc = __shfl(gz, 4 * lr, 64);
    }
    if constexpr (MODE == kDkv) {
      load_tile(p, a.v + kbase, row0, N, l);
      put_natural<L::LN>(nat, p, l);
    }
    __syncthreads();
    if constexpr (!kSums) f2 = read_row<L::LN>(nat, l);
  }
  Blk<F32> f1[GP];
  int wo[GP];
#pragma unroll
  for (int g = 0; g < GP; ++g) {
    f1[g] = fixed_window(&sh.fixed[lr][0], hd.at[g], hd.count[g], l);
    wo[g] = window_offset<F32, GP>(hd.at[g], l);
  }
  const bool any_more = hd.any_more;
  wave_order();

  f32x4 acc[MODE == kDkv ? 4 : 1] = {};  // dv columns (dkv)
  f32x4 gacc[kSums ? 4 : GP + kMore] = {};  // num or dv columns; else the groups' gradient blocks
  float z = 0.f;
  float co[MODE == kDq ? coef_count(GP) : 1];
#pragma unroll
  for (int x = 0; x < (MODE == kDq ? coef_count(GP) : 1); ++x) co[x] = 0.f;
  const bool want_grad = MODE == kDkv || (MODE == kDq && a.dq), want_co = MODE == kDq && a.part;
  const int fc = row0 + lr;  // the lane's fixed token
  const T* const s1 = kKeys ? a.q + qbase : a.k + kbase;
  auto load_second = [&](auto& p, int r0) {
    if constexpr (kKeys)
      load_tile(p, const_cast<const E*>(a.Gv) + qbase, r0, N, l);
    else
      load_tile(p, a.v + kbase, r0, N, l);
  };
  const int begin = (kKeys ? ft : 0) + wave;
  const int end = kSums || want_grad || want_co ? (kKeys ? NT : ft + 1) : 0;
  Piece<T> p1;
  std::conditional_t<kKeys, Piece<E>, Piece<T>> p2;
  if (begin < end) {
    load_tile(p1, s1, begin * kM, N, l);
    load_second(p2, begin * kM);
  }
  for (int st = begin; st < end; st += kWv) {
    put_sorted(&sh.sorted[0][0][0], p1, off);
    put_natural<L::LN>(nat, p2, l);
    wave_order();
    if (st + kWv < end) {  // the next tile's rows, in flight during this one
      load_tile(p1, s1, (st + kWv) * kM, N, l);
      load_second(p2, (st + kWv) * kM);
    }
    // pairs [streamed 4 lg + r][fixed lr]
    f32x4 s[GP];
#pragma unroll
    for (int g = 0; g < GP; ++g) s[g] = mma(read_at<F32>(srt, wo[g]), f1[g], f32x4{});
    if (any_more) {
      // A scalar branch a slot and a group. As selects of all groups over all slots,
      // present or not, it was 190 VALU instructions a tile: B=2, N=1000, 14 heads, sizes
      // 22 and seven of 6, forward 54 us, 44 now (37 with no group beyond 16 dimensions),
      // fp32 forward and backward 664, 536 now. Unrolled, it takes 50 more registers.
#pragma unroll 1
      for (int m = 0; m < kMore; ++m) {
        const Window w = more_window(sh.more, m);
        if (!w.present()) continue;
        const Blk<F32> a1 = read_window<F32>(srt + lr * L::LS, w.at(), l),
                       b1 = fixed_window(&sh.fixed[lr][0], w.at(), w.count(), l);
#pragma unroll
        for (int g = 0; g < GP; ++g)
          if (w.group() == g) s[g] = mma(a1, b1, s[g]);
      }
    }
    // tiles off the diagonal and inside the sequence: every pair counts
    const bool edge = kKeys ? st <= ft || (st + 1) * kM > N : st >= ft;
    auto mask = [&](f32x4& x) {
      if (!edge) return;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int sc = st * kM + 4 * lg + r;
        x[r] = (kKeys ? fc <= sc && sc < N && fc < N : sc <= fc && sc < N) ? x[r] : 0.f;
      }
    };
    f32x4 ds = {};
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int sc = st * kM + 4 * lg + r;
      if constexpr (MODE == kDkv) ds[r] = a.Gz[(size_t)bh * N + (sc < N ? sc : N - 1)];
      if constexpr (MODE == kDq) ds[r] = gzc;
    }
    if constexpr (!kSums) {
      ds = mma(read_row<L::LN>(nat, l), f2, ds);
      mask(ds);
    }
    if constexpr (kSums) {
      f32x4 kap;
#pragma unroll
      for (int r = 0; r < 4; ++r) kap[r] = kappa_of<GP>(cf, s, r);
      mask(kap);
#pragma unroll
      for (int r = 0; r < 4; ++r) z += kap[r];
      if constexpr (F32) {
        const Blk<F32> ka = as_operand<F32>(kap);
#pragma unroll
        for (int cb = 0; cb < 4; ++cb) gacc[cb] = mma(ka, rows_operand(nat, L::LN, 16 * cb, lr, l), gacc[cb]);
      } else {
        // kappa in two parts. One rounds it to 2^-9, on evenly scaled inputs more than the
        // state route loses in its features' many independent roundings: at N=800, 8 groups
        // num's error was 1.7e-3 and dv's, of an upstream of num, 2.9e-3, against the
        // state's 1.5e-3 and 2.7e-3; in two parts 2.6e-6 and 2.3e-3 (dv's own type and
        // G's). They cost up to 4 % of a forward (B=2, N=1000 36.8 to 38.1 us) and up to 2 %
        // of a forward and backward (205 to 209).
        const float y[4] = {kap[0], kap[1], kap[2], kap[3]};
        Blk<F32> ka[2];
        s16x4 parts[2];
        split4(parts, y);
        ka[0].v = parts[0];
        ka[1].v = parts[1];
#pragma unroll
        for (int cb = 0; cb < 4; ++cb) {
          const Blk<F32> vb = rows_operand(nat, L::LN, 16 * cb, lr, l);
          gacc[cb] = mma(ka[0], vb, gacc[cb]);
          gacc[cb] = mma(ka[1], vb, gacc[cb]);
        }
      }
    }
    if (want_co) {
      if constexpr (MODE == kDq) {
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          co[0] += ds[r];
#pragma unroll
          for (int g = 0; g < GP; ++g) {
            const float x = ds[r] * s[g][r];
            co[1 + g] += x;
#pragma unroll
            for (int y = 0; y <= g; ++y)
              co[1 + GP + g * (g + 1) / 2 + y] = fmaf(x, s[y][r], co[1 + GP + g * (g + 1) / 2 + y]);
          }
        }
      }
    }
    if constexpr (!kSums) {
      if (want_grad) {
        f32x4 kap = {2.f * cf.c0, 2.f * cf.c0, 2.f * cf.c0, 2.f * cf.c0};  // twice kappa
        Window w[kMore];
        if (any_more) {
#pragma unroll
          for (int m = 0; m < kMore; ++m) w[m] = more_window(sh.more, m);
        }
#pragma unroll
        for (int g = 0; g < GP; ++g) {
          f32x4 x;
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const float t = slope<GP>(cf, s, g, r);
            if constexpr (MODE == kDkv) kap[r] = fmaf(s[g][r], cf.lin[g] + t, kap[r]);
            x[r] = ds[r] * t;
          }
          const Blk<F32> xa = as_operand<F32>(x);
          gacc[g] = mma(xa, rows_operand(srt, L::LS, hd.at[g], L::in_block(lr), l), gacc[g]);
          if (any_more) {
#pragma unroll
            for (int m = 0; m < kMore; ++m)
              if (w[m].group() == g)
                gacc[GP + m] = mma(xa, rows_operand(srt, L::LS, 16 * (GP + m), L::in_block(lr), l), gacc[GP + m]);
          }
        }
        if constexpr (MODE == kDkv) {
          kap *= 0.5f;
          mask(kap);
          const Blk<F32> ka = as_operand<F32>(kap);
#pragma unroll
          for (int cb = 0; cb < 4; ++cb) acc[cb] = mma(ka, rows_operand(nat, L::LN, 16 * cb, lr, l), acc[cb]);
        }
      }
    }
    wave_order();
  }

  // the waves' sums, in wave order, through LDS tiles of [16][64] floats
  __syncthreads();
  static_assert(sizeof(sh.sorted) >= 2 * kM * kD * sizeof(float), "the epilogue's tiles reuse the sorted tiles");
  float* const t0 = reinterpret_cast<float*>(&sh.sorted[0][0][0]);
  float* const t1 = t0 + kM * kD;
  if constexpr (MODE == kFwd) {
    z += __shfl_xor(z, 16, 64);
    z += __shfl_xor(z, 32, 64);
    if (lg == 0) sh.zrow[wave][lr] = z;
  }
  if constexpr (MODE == kDq) {
    if (want_co) {
#pragma unroll
      for (int x = 0; x < coef_count(GP); ++x) {
        const float y = wave_sum(co[x]);
        if (l == 0) sh.co[wave][x] = y;
      }
    }
  }
  in_wave_order(wave, [&](bool fresh) {
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      float* const row = t0 + (4 * lg + r) * kD;
      if constexpr (kSums) {
#pragma unroll
        for (int cb = 0; cb < 4; ++cb) row[16 * cb + lr] = gacc[cb][r] + (fresh ? 0.f : row[16 * cb + lr]);
      } else {
#pragma unroll
        for (int g = 0; g < GP + kMore; ++g) {
          const int d = sh.dim[16 * g + lr];
          if (d < kD) row[d] = gacc[g][r] + (fresh ? 0.f : row[d]);
        }
      }
      if constexpr (MODE == kDkv) {
        float* const row1 = t1 + (4 * lg + r) * kD;
#pragma unroll
        for (int cb = 0; cb < 4; ++cb) row1[16 * cb + lr] = acc[cb][r] + (fresh ? 0.f : row1[16 * cb + lr]);
      }
    }
  });
  if constexpr (MODE == kDq) {
    if (want_co && threadIdx.x < coef_count(GP)) {
      float y = 0.f;
#pragma unroll
      for (int w = 0; w < kWv; ++w) y += sh.co[w][threadIdx.x];
      a.part[((size_t)bh * NT + ft) * coef_count(GP) + threadIdx.x] = y;
    }
  }
  // one 4-wide piece of a row per thread
  const int er = threadIdx.x >> 4, ec = 4 * (threadIdx.x & 15), tok = row0 + er;
  if (tok >= N) return;
  const float4 x = *reinterpret_cast<const float4*>(t0 + er * kD + ec);
  if constexpr (MODE == kFwd) {
    float zz = 0.f;
#pragma unroll
    for (int w = 0; w < kWv; ++w) zz += sh.zrow[w][er];
    const float dp = a.floor > 0.f ? fmaxf(zz, a.floor) : zz;
    const size_t o = qbase + (size_t)tok * kD + ec;
    *reinterpret_cast<float4*>(a.num + o) = x;
    store4(a.out + o, make_float4(x.x / dp, x.y / dp, x.z / dp, x.w / dp));
    if (ec == 0) a.den[(size_t)bh * N + tok] = zz;
  }
  if constexpr (MODE == kDq) {
    if (a.dq) store4(a.dq + qbase + (size_t)tok * kD + ec, x);
  }
  if constexpr (MODE == kDkv) {
    const size_t o = qbase + (size_t)tok * kD + ec;
    *reinterpret_cast<float4*>(a.dkh + o) = x;
    *reinterpret_cast<float4*>(a.dvh + o) = *reinterpret_cast<const float4*>(t1 + er * kD + ec);
  }
  if constexpr (MODE == kDv) *reinterpret_cast<float4*>(a.dvh + qbase + (size_t)tok * kD + ec) = x;
}

template <typename T, bool F32, int GP, int MODE>
__global__ __launch_bounds__(64 * kWv, 2) void direct_tiles(const Args<T, F32> a) {
  __shared__ __attribute__((aligned(16))) Shared<F32, GP> sh;
  tiles<T, F32, GP, MODE>(a, sh);
}

// ---------------------------------------------------------------------------
// bf16 backward. dq_i[d] = sum_h c_h(d) P_h[i][d] over h = 0 .. GP (s_GP = 1) with
//   P_h[i][d] = sum_j (ds s_h) k_j[d],  c_h(d) = 2 A_g(d)h, c_GP(d) = a_g(d):
// the sums over keys stay in the matrix cores' accumulators for the whole row,
// and the quadratic form and the coefficient sums
//   sum ds s_g s_h = sum_i sum_{d in g} q_i[d] P_h[i][d]
// are applied once at its end. A tile's VALU work is then ds s_h alone, 36
// multiplies and their packs a lane against about 560 instructions with the slopes
// t_g and the 45 coefficient products formed per pair. For the coefficient sums ds
// s_h goes in as several bf16 parts (as one, their error was 1.07 to 1.14 times as
// large as that of fp32 sums over the pairs up to N = 256). Three up to kC
// tokens, where the state route sums fp32 pair values: with an upstream of den
// alone G is zero and ds exact, and two parts gave lam's gradient 2.5e-6 where
// those sums give 1e-7. Two beyond, where that route's state holds bf16 features
// (1e-3). dk likewise, with the streamed q and one part; dv needs kappa, formed as
// in the forward (tiles).
//
// All (GP + 1) x 4 column blocks of P are 144 registers, too many for one wave,
// and P_h needs s_h alone: the four waves share each staged step of 64 streamed
// rows and wave w takes the groups w GP / 4 .. and column block w of P_GP. Two
// tiles of a step make one 32-deep product (k slots 8 g + 0 .. 3 the first tile's rows 4 g .., + 4
// .. 7 the second's).
// ---------------------------------------------------------------------------
__device__ __forceinline__ bf16x8 both(s16x4 a, s16x4 b) {
  return __builtin_bit_cast(bf16x8, __builtin_shufflevector(a, b, 0, 1, 2, 3, 4, 5, 6, 7));
}
template <int GP>
struct SharedRoles {
  using L = Lay<false, GP>;
  union {
    struct {
      uint16_t sorted[kStep][L::LS];
      uint16_t nat1[kStep][L::LN], nat2[kStep][L::LN];  // k and v, or q and G
    };
    struct {
      float t0[kM][kD];     // results
      float y[GP + 1][kD];  // coefficient sums per dimension
    };
  };
  uint16_t fixed[kM][L::LS];
  uint16_t fnat[kM][L::LN];  // dq: q
  float gz[kStep];           // dk: Gz of the step's rows
  int grp[kD];               // dq: group of a dimension
  uint32_t more[kMore];
  float dc0[kWv];
};

template <typename T, int GP, int MODE, int PARTS>
__device__ __forceinline__ void roles(const Args<T, false>& a, SharedRoles<GP>& sh) {
  using L = Lay<false, GP>;
  constexpr int kOwn = GP / kWv;  // groups per wave
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), l = threadIdx.x & 63, lr = l & 15, lg = l >> 4;
  const int NT = gridDim.y, bh = blockIdx.x, N = a.N;
  // longest first, of all heads (B=2, N=1000, 14 heads: dq 110 to 87 us, dk and dv 113 to 97)
  const int ft = MODE == kDk ? (int)blockIdx.y : NT - 1 - (int)blockIdx.y;
  const int R = a.Hq / a.Hkv, b = bh / a.Hq, h = bh % a.Hq, u = b * a.Hkv + h / R;
  const size_t qbase = (size_t)bh * N * kD, kbase = (size_t)u * N * kD;
  const int row0 = ft * kM;

  const Head<false, GP> hd = read_head<false, GP>(a.labels, a.lam, a.gam, a.G, h, a.scale, l, sh.more);
  zero_lds(sh.sorted);
  zero_lds(sh.fixed);
  if (MODE == kDq && wave == 0) sh.grp[l] = hd.lab;
  int off[16];
  piece_offsets(off, hd, wave * kM, l);
  __syncthreads();
  Row<false> f2;
  float gzc = 0.f;
  {
    Piece<T> p;
    load_tile(p, MODE == kDk ? a.k + kbase : a.q + qbase, row0, N, l);
    if (wave == 0) put_sorted(&sh.fixed[0][0], p, off);
    if constexpr (MODE == kDq) {
      if (wave == 0) put_natural<L::LN>(&sh.fnat[0][0], p, l);
      Piece<uint16_t> gp;
      float gz;
      normalization_vjp<T, false>(gp, gz, a, bh, row0, wave, l);
      if (wave == 0) put_natural<L::LN>(&sh.nat2[0][0], gp, l);
      gzc = __shfl(gz, 4 * lr, 64);
    } else {
      load_tile(p, a.v + kbase, row0, N, l);
      if (wave == 0) put_natural<L::LN>(&sh.nat2[0][0], p, l);
    }
    __syncthreads();
    f2 = read_row<L::LN>(&sh.nat2[0][0], l);
  }
  // the wave's own groups
  Blk<false> fo[kOwn];
  int wown[kOwn];
#pragma unroll
  for (int x = 0; x < kOwn; ++x) {
    int at = hd.at[x], n = hd.count[x];
#pragma unroll
    for (int w = 1; w < kWv; ++w) {
      at = wave == w ? hd.at[w * kOwn + x] : at;
      n = wave == w ? hd.count[w * kOwn + x] : n;
    }
    fo[x] = fixed_window(&sh.fixed[lr][0], at, n, l);
    wown[x] = window_offset<false, GP>(at, l);
  }
  // and the further windows: place among the wave's own groups, fixed operand, offset.
  // They all fall to the waves whose groups are long while the others wait, so their
  // reads go out together (one head of 2400 tokens, sizes 57 and seven of 1, forward and
  // backward 288 us read one after the other, 217 so)
  int xm[kMore], wm[kMore];
  Blk<false> fm[kMore];
  bool own_more = false;
#pragma unroll
  for (int m = 0; m < kMore; ++m) {
    const Window w = more_window(sh.more, m);
    xm[m] = w.group() - wave * kOwn;
    own_more |= xm[m] >= 0 && xm[m] < kOwn;
    fm[m] = fixed_window(&sh.fixed[lr][0], w.at(), w.count(), l);
    wm[m] = window_offset<false, GP>(w.at(), l);
  }
  f32x4 P[kOwn][4] = {}, Pl = {};
  float c0sum = 0.f;
  const int fc = row0 + lr;
  const bool want = MODE == kDk || a.dq || a.part;
  const int begin = MODE == kDk ? ft / 4 : 0, end = want ? (MODE == kDk ? (NT + 3) / 4 : ft / 4 + 1) : 0;
  const T* const s1 = MODE == kDk ? a.q + qbase : a.k + kbase;
  Piece<T> p1;
  std::conditional_t<MODE == kDk, Piece<uint16_t>, Piece<T>> p2;
  float pz = 0.f;
  auto fetch = [&](int step) {
    const int r0 = step * kStep + wave * kM;
    load_tile(p1, s1, r0, N, l);
    if constexpr (MODE == kDk) {
      load_tile(p2, const_cast<const uint16_t*>(a.Gv) + qbase, r0, N, l);
      const int row = r0 + lr;
      pz = a.Gz[(size_t)bh * N + (row < N ? row : N - 1)];
    } else {
      load_tile(p2, a.v + kbase, r0, N, l);
    }
  };
  if (begin < end) fetch(begin);
  for (int step = begin; step < end; ++step) {
    lds_sync();  // the previous step's reads (and the prologue's)
    put_sorted(&sh.sorted[0][0], p1, off);
    put_natural<L::LN>(&sh.nat1[wave * kM][0], p1, l);
    put_natural<L::LN>(&sh.nat2[wave * kM][0], p2, l);
    if constexpr (MODE == kDk) {
      if (lg == 0) sh.gz[wave * kM + lr] = pz;
    }
    lds_sync();
    if (step + 1 < end) fetch(step + 1);
    const int t0 = step * 4;  // the step's tiles
#pragma unroll 1
    for (int pr = 0; pr < 2; ++pr) {
      const int ta = t0 + 2 * pr;
      if (MODE == kDk ? ta + 1 < ft || ta >= NT : ta > ft) continue;
      s16x4 xh[2][kOwn][PARTS], xl[2][PARTS];  // of ds s_h and ds
#pragma unroll
      for (int e = 0; e < 2; ++e) {
        const int r0 = (2 * pr + e) * kM, tok = (ta + e) * kM + 4 * lg;
        f32x4 ds;
        if constexpr (MODE == kDk) {
          ds = *reinterpret_cast<const f32x4*>(&sh.gz[r0 + 4 * lg]);
        } else {
          ds = f32x4{gzc, gzc, gzc, gzc};
        }
        ds = mma(read_row<L::LN>(&sh.nat2[r0][0], l), f2, ds);
        f32x4 s[kOwn];
#pragma unroll
        for (int x = 0; x < kOwn; ++x)
          s[x] = mma(read_at<false>(&sh.sorted[r0][0], wown[x]), fo[x], f32x4{});
        if (own_more) {
          Blk<false> a1[kMore];
#pragma unroll
          for (int m = 0; m < kMore; ++m) a1[m] = read_at<false>(&sh.sorted[r0][0], wm[m]);
#pragma unroll
          for (int m = 0; m < kMore; ++m) {
            const f32x4 e = mma(a1[m], fm[m], f32x4{});
#pragma unroll
            for (int x = 0; x < kOwn; ++x)
              if (xm[m] == x) {
#pragma unroll
                for (int r = 0; r < 4; ++r) s[x][r] += e[r];
              }
          }
        }
        float y[4] = {ds[0], ds[1], ds[2], ds[3]};
        if (MODE == kDk ? ta + e <= ft || (ta + e + 1) * kM > N : ta + e >= ft) {  // else every pair counts
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const bool ok = MODE == kDk ? fc <= tok + r && tok + r < N && fc < N : tok + r <= fc && tok + r < N;
            y[r] = ok ? y[r] : 0.f;
          }
        }
        if (MODE == kDq && ((ta + e) & 3) == wave) c0sum += (y[0] + y[1]) + (y[2] + y[3]);
        split4(xl[e], y);
#pragma unroll
        for (int x = 0; x < kOwn; ++x) {
          const float z[4] = {y[0] * s[x][0], y[1] * s[x][1], y[2] * s[x][2], y[3] * s[x][3]};
          split4(xh[e][x], z);
        }
      }
      const uint16_t* const ka = &sh.nat1[2 * pr * kM][0];
      const uint16_t* const kb = &sh.nat1[(2 * pr + 1) * kM][0];
      auto operand = [&](int col0) {
        return both(rows_operand(ka, L::LN, col0, 0, l).v, rows_operand(kb, L::LN, col0, 0, l).v);
      };
#pragma unroll
      for (int cb = 0; cb < 4; ++cb) {
        const bf16x8 k8 = operand(16 * cb);
#pragma unroll
        for (int x = 0; x < kOwn; ++x)
#pragma unroll
          for (int f = 0; f < PARTS; ++f) P[x][cb] = mfma16(both(xh[0][x][f], xh[1][x][f]), k8, P[x][cb]);
      }
      const bf16x8 kl = operand(16 * wave);
#pragma unroll
      for (int f = 0; f < PARTS; ++f) Pl = mfma16(both(xl[0][f], xl[1][f]), kl, Pl);
    }
  }

  // the waves' parts in wave order, through LDS
  __syncthreads();
  in_wave_order(wave, [&](bool fresh) {
#pragma unroll
    for (int cb = 0; cb < 4; ++cb) {
      const int d = 16 * cb + lr, gd = __shfl(hd.lab, d, 64);
      float c[kOwn];
#pragma unroll
      for (int x = 0; x < kOwn; ++x) c[x] = 2.f * __shfl(hd.gam, 8 * gd + wave * kOwn + x, 64);
      const float cl = cb == wave ? __shfl(hd.lam, gd, 64) : 0.f;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        float v = fresh ? 0.f : sh.t0[4 * lg + r][d];
#pragma unroll
        for (int x = 0; x < kOwn; ++x) v = fmaf(c[x], P[x][cb][r], v);
        sh.t0[4 * lg + r][d] = fmaf(cl, Pl[r], v);
      }
    }
  });
  if constexpr (MODE == kDq) {
    if (a.part) {
      // sum over the tile's queries of q_i[d] P_h[i][d]
#pragma unroll
      for (int cb = 0; cb < 4; ++cb) {
        float qv[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) qv[r] = bf16_to_f(sh.fnat[4 * lg + r][16 * cb + lr]);
        auto put = [&](int hh, const f32x4& p) {
          float y = qv[0] * p[0];
#pragma unroll
          for (int r = 1; r < 4; ++r) y = fmaf(qv[r], p[r], y);
          y += __shfl_xor(y, 16, 64);
          y += __shfl_xor(y, 32, 64);
          if (lg == 0) sh.y[hh][16 * cb + lr] = y;
        };
#pragma unroll
        for (int x = 0; x < kOwn; ++x) put(wave * kOwn + x, P[x][cb]);
        if (cb == wave) put(GP, Pl);
      }
      c0sum = wave_sum(c0sum);
      if (l == 0) sh.dc0[wave] = c0sum;
      __syncthreads();
      constexpr int kCo = role_coef_count(GP);
      float* const dst = a.part + ((size_t)bh * NT + ft) * kCo;
      const int t = threadIdx.x;
      if (t < (GP + 1) * GP) {
        const int hh = t / GP, g = t % GP;
        float y = 0.f;
#pragma unroll 1
        for (int d0 = 0; d0 < kD; d0 += 16) {
          float v[16];
          int o[16];
#pragma unroll
          for (int d = 0; d < 16; ++d) {
            v[d] = sh.y[hh][d0 + d];
            o[d] = sh.grp[d0 + d];
            asm volatile("" : "+v"(v[d]));  // read whether or not it counts, not behind a branch
          }
#pragma unroll
          for (int d = 0; d < 16; ++d) y += o[d] == g ? v[d] : 0.f;
        }
        dst[1 + t] = y;
      }
      if (t == 0) dst[0] = (sh.dc0[0] + sh.dc0[1]) + (sh.dc0[2] + sh.dc0[3]);
    }
  }
  const int er = threadIdx.x >> 4, ec = 4 * (threadIdx.x & 15), tok = row0 + er;
  if (tok >= N) return;
  const size_t o = qbase + (size_t)tok * kD + ec;
  const float4 x = *reinterpret_cast<const float4*>(&sh.t0[er][ec]);
  if constexpr (MODE == kDq) {
    if (a.dq) store4(a.dq + o, x);
  } else {
    *reinterpret_cast<float4*>(a.dkh + o) = x;
  }
}

template <typename T, int GP, int PARTS>
__global__ __launch_bounds__(64 * kWv, 3) void direct_dq(const Args<T, false> a) {
  __shared__ __attribute__((aligned(16))) SharedRoles<GP> sh;
  roles<T, GP, kDq, PARTS>(a, sh);
}

// dk in the blocks of z = 0, dv in those of z = 1: side by side their chains
// overlap, and each needs fewer registers than one kernel of both (201 and two
// waves per SIMD).
template <typename T, int GP>
__global__ __launch_bounds__(64 * kWv, 3) void direct_dk_dv(const Args<T, false> a) {
  __shared__ __attribute__((aligned(16))) union {
    SharedRoles<GP> k;
    Shared<false, GP> v;
  } sh;
  if (blockIdx.z == 0)
    roles<T, GP, kDk, 1>(a, sh.k);
  else
    tiles<T, false, GP, kDv>(a, sh.v);
}

// The last launch of a backward: blocks [0, sums) add the unit's R heads of dk
// and dv in head order (four values a thread); blocks beyond add the
// coefficient sums of one head over (batch, tile) in a fixed order and write
// dc0, dlam and the symmetric dgam.
template <typename T, bool F32, int GP>
__global__ __launch_bounds__(256) void direct_finish(const float* __restrict__ dkh, const float* __restrict__ dvh, int R,
                                                     size_t per_head, size_t total4, int sums, T* __restrict__ dk,
                                                     T* __restrict__ dv, const float* __restrict__ part, int B, int Hq,
                                                     int NT, int G, float scale, float* __restrict__ dc0,
                                                     float* __restrict__ dlam, float* __restrict__ dgam) {
  if ((int)blockIdx.x < sums) {
    const size_t x = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (x >= total4) return;
    const size_t e = 4 * x;
    const size_t at = (e / per_head) * R * per_head + e % per_head;
    float4 k4 = make_float4(0.f, 0.f, 0.f, 0.f), v4 = k4;
#pragma unroll 4
    for (int r = 0; r < R; ++r) {
      const float4 y = *reinterpret_cast<const float4*>(dkh + at + (size_t)r * per_head);
      const float4 w = *reinterpret_cast<const float4*>(dvh + at + (size_t)r * per_head);
      k4.x += y.x;
      k4.y += y.y;
      k4.z += y.z;
      k4.w += y.w;
      v4.x += w.x;
      v4.y += w.y;
      v4.z += w.z;
      v4.w += w.w;
    }
    if (dk) store4(dk + e, k4);
    if (dv) store4(dv + e, v4);
    return;
  }
  constexpr int kCo = F32 ? coef_count(GP) : role_coef_count(GP);
  __shared__ float w[kCo];
  // row groups of kCo columns read together, eight rows in flight a thread
  constexpr int kRows = 256 / kCo;
  __shared__ float wr[kRows][kCo];
  const int h = blockIdx.x - sums, c = threadIdx.x % kCo, rg = threadIdx.x / kCo, rows = B * NT;
  if (rg < kRows) {
    float x = 0.f;
    for (int i0 = rg; i0 < rows; i0 += 8 * kRows) {
      float y[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const int i = min(i0 + e * kRows, rows - 1);
        y[e] = part[((size_t)(i / NT * Hq + h) * NT + i % NT) * kCo + c];
      }
#pragma unroll
      for (int e = 0; e < 8; ++e) x += i0 + e * kRows < rows ? y[e] : 0.f;
    }
    wr[rg][c] = x;
  }
  __syncthreads();
  if (threadIdx.x < kCo) {
    float x = wr[0][threadIdx.x];
#pragma unroll
    for (int r = 1; r < kRows; ++r) x += wr[r][threadIdx.x];
    w[threadIdx.x] = x;
  }
  __syncthreads();
  if (threadIdx.x == 0) dc0[h] = w[0];
  for (int e = threadIdx.x; e < G; e += 256) dlam[(size_t)h * G + e] = scale * w[F32 ? 1 + e : 1 + GP * GP + e];
  for (int e = threadIdx.x; e < G * G; e += 256) {
    const int x = e / G, y = e % G, hi = x > y ? x : y, lo = x > y ? y : x;
    // bf16: the two ways round differ by the rounding of ds s_h
    const float y2 = F32 ? w[1 + GP + hi * (hi + 1) / 2 + lo] : 0.5f * (w[1 + hi * GP + lo] + w[1 + lo * GP + hi]);
    dgam[(size_t)h * G * G + e] = scale * scale * y2;
  }
}

// ---------------------------------------------------------------------------
// Host launches.
// ---------------------------------------------------------------------------
namespace {

template <bool F32>
struct Work {
  Elem<F32>* Gv;
  float *Gz, *dkh, *dvh, *part;
  size_t bytes;
};
template <bool F32>
Work<F32> work_of(void* base, int B, int Hq, int N) {
  char* p = static_cast<char*>(base);
  size_t used = 0;
  auto take = [&](size_t n) {
    char* x = p ? p + used : nullptr;
    used += align256(n);
    return x;
  };
  const size_t rows = (size_t)B * Hq * N;
  Work<F32> w;
  w.Gv = reinterpret_cast<Elem<F32>*>(take(sizeof(Elem<F32>) * rows * kD));
  w.Gz = reinterpret_cast<float*>(take(sizeof(float) * rows));
  w.dkh = reinterpret_cast<float*>(take(sizeof(float) * rows * kD));
  w.dvh = reinterpret_cast<float*>(take(sizeof(float) * rows * kD));
  w.part = reinterpret_cast<float*>(
      take(sizeof(float) * (size_t)B * Hq * ((N + kM - 1) / kM) * (F32 ? coef_count(8) : role_coef_count(8))));
  w.bytes = used;
  return w;
}

template <typename T, bool F32, int GP>
void backward_of(const LaunchGeom& g, const Args<T, F32>& a, const Work<F32>& w, T* dk, T* dv, float* dc0, float* dlam,
                 float* dgam, hipStream_t st, const Timer& timed) {
  const int NT = (g.N + kM - 1) / kM;
  const dim3 grid(g.B * g.Hq, NT), block(64 * kWv);
  const bool kv = dk || dv;
  if constexpr (F32) {
    timed("direct_dq", st, [&] { hipLaunchKernelGGL((direct_tiles<T, true, GP, kDq>), grid, block, 0, st, a); });
    if (kv)
      timed("direct_dkv", st, [&] { hipLaunchKernelGGL((direct_tiles<T, true, GP, kDkv>), grid, block, 0, st, a); });
  } else {
    timed("direct_dq", st, [&] {
      if (g.N <= kC)
        hipLaunchKernelGGL((direct_dq<T, GP, 3>), grid, block, 0, st, a);
      else
        hipLaunchKernelGGL((direct_dq<T, GP, 2>), grid, block, 0, st, a);
    });
    if (kv)
      timed("direct_dkv", st,
            [&] { hipLaunchKernelGGL((direct_dk_dv<T, GP>), dim3(grid.x, grid.y, 2), block, 0, st, a); });
  }
  const size_t per_head = (size_t)g.N * kD, total4 = (size_t)g.B * g.Hkv * per_head / 4;
  const int sums = kv ? (int)((total4 + 255) / 256) : 0, heads = dc0 ? g.Hq : 0;
  if (sums + heads)
    timed("direct_finish", st, [&] {
      hipLaunchKernelGGL((direct_finish<T, F32, GP>), dim3(sums + heads), dim3(256), 0, st, w.dkh, w.dvh, g.R, per_head,
                         total4, sums, dk, dv, w.part, g.B, g.Hq, NT, a.G, a.scale, dc0, dlam, dgam);
    });
}

}  // namespace

size_t direct_work_bytes(bool f32, int B, int Hq, int N) {
  return f32 ? work_of<true>(nullptr, B, Hq, N).bytes : work_of<false>(nullptr, B, Hq, N).bytes;
}

template <typename T, bool F32>
void launch_direct_forward(const LaunchGeom& g, const T* q, const T* k, const T* v, const int32_t* labels,
                           const float* c0, const float* lam, const float* gam, int groups, float scale, float floor,
                           T* out, float* num, float* den, hipStream_t st, const Timer& timed) {
  Args<T, F32> a{q, k, v, labels, c0, lam, gam, groups, g.Hq, g.Hkv, g.N, scale, floor, out, num, den};
  const dim3 grid(g.B * g.Hq, (g.N + kM - 1) / kM), block(64 * kWv);
  timed("direct_fwd", st, [&] {
    if (groups <= 4)
      hipLaunchKernelGGL((direct_tiles<T, F32, 4, kFwd>), grid, block, 0, st, a);
    else
      hipLaunchKernelGGL((direct_tiles<T, F32, 8, kFwd>), grid, block, 0, st, a);
  });
}

template <typename T, bool F32>
void launch_direct_backward(const LaunchGeom& g, const T* q, const T* k, const T* v, const int32_t* labels,
                            const float* c0, const float* lam, const float* gam, int groups, float scale, float floor,
                            const float* num, const float* den, const T* dout, const float* dnum, const float* dden,
                            T* dq, T* dk, T* dv, float* dc0, float* dlam, float* dgam, void* workspace, hipStream_t st,
                            const Timer& timed) {
  const Work<F32> w = work_of<F32>(workspace, g.B, g.Hq, g.N);
  Args<T, F32> a{q, k, v, labels, c0, lam, gam, groups, g.Hq, g.Hkv, g.N, scale, floor, nullptr,
                 const_cast<float*>(num), const_cast<float*>(den), dout, dnum, dden, w.Gv, w.Gz, dq,
                 dc0 ? w.part : nullptr, w.dkh, w.dvh};
  if (groups <= 4)
    backward_of<T, F32, 4>(g, a, w, dk, dv, dc0, dlam, dgam, st, timed);
  else
    backward_of<T, F32, 8>(g, a, w, dk, dv, dc0, dlam, dgam, st, timed);
}

#define OAL_DIRECT(T, F32)                                                                                             \
  template void launch_direct_forward<T, F32>(const LaunchGeom&, const T*, const T*, const T*, const int32_t*,         \
                                              const float*, const float*, const float*, int, float, float, T*, float*, \
                                              float*, hipStream_t, const Timer&);                                      \
  template void launch_direct_backward<T, F32>(const LaunchGeom&, const T*, const T*, const T*, const int32_t*,        \
                                               const float*, const float*, const float*, int, float, float,            \
                                               const float*, const float*, const T*, const float*, const float*, T*,   \
                                               T*, T*, float*, float*, float*, void*, hipStream_t, const Timer&);
OAL_DIRECT(uint16_t, false)
OAL_DIRECT(uint16_t, true)
OAL_DIRECT(float, false)
OAL_DIRECT(float, true)
#undef OAL_DIRECT

}  // namespace oal
