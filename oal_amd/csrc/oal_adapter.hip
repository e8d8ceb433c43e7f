// Small kernels around the operator for gfx950: what a call of the public entry
// points needs besides the attention itself, each in one launch.
//
//   k_expand_factor      packed lower-triangular factor L -> c0 = M_00 + eps,
//                        lam = 2 M_0,1.., gam = M_1..,1.. with M = L L^T
//                        (reference grouped_quadratic.py:184-218)
//   k_expand_factor_bwd  its VJP, dL = (dM + dM^T) L on the lower triangle
//   k_expand_pairs       per-pair coefficients c [Hq][D (D + 1) / 2] -> the symmetric
//                        gam [Hq][64][64], b -> lam, and the labels d -> d
//   k_expand_pairs_bwd   dgam -> dc (an off-diagonal pair has two entries)
//   k_check_labels       group labels -> int32 [Hq][64], and whether they are valid
//                        (reference grouped_quadratic.py:136-181)
//   k_check_outputs      whether num, den and out are finite and den positive
//                        (reference grouped_quadratic.py:379-397,
//                        hd_block_gemm_runtime.py:392-408)
//
//   k_rotary_heads       projections [B][N][heads 64] of q, k, v -> head-first [B][heads]
//                        [N][64], q and k rotated (rotate-half rotary embedding,
//                        reference qwen_lora_experiment/attention/common.py:510-596);
//                        and back, for the gradients
//
// The rotation and the three transposes took 13 launches forward and 16 backward,
// several passes over q each; in one pass it is bound by memory at large sizes and by
// its launch below. The pair kernels took 12 launches as torch operations (index gathers and
// scatters, 50 us of kernels beside 330 us for the operator at N = 1024).
// All are bound by their launch: a few hundred values, or one pass over the
// outputs. As torch operations the expansion took 14 launches and its VJP about 20,
// the checks 3 to 14 launches with 2 to 5 host synchronizations, 190 us of host
// time in a forward of 266 us at N = 128. A check writes its verdict into a
// host-mapped word only when something is wrong, so the host needs one
// synchronization and no copy.

#include <hip/hip_fp16.h>
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <algorithm>

#include "oal_common.hpp"
#include "oal_internal.hpp"

namespace oal {

namespace {

constexpr int kSideMax = kD + 1;
constexpr int kPackMax = kSideMax * (kSideMax + 1) / 2;
constexpr int kThreads = 256;

__device__ __forceinline__ int packed(int i, int m) { return i * (i + 1) / 2 + m; }

}  // namespace

// One block per query head, the sums in fp64 (a few hundred terms, no time). M[i][j] and M[j][i] are the same sum in the same
// order, so gam is exactly symmetric (the intra-chunk kernels rely on it).
template <typename T>
__global__ __launch_bounds__(kThreads) void k_expand_factor(const T* __restrict__ factor, bool per_head, int G, T eps,
                                                            T* __restrict__ c0, T* __restrict__ lam,
                                                            T* __restrict__ gam) {
  __shared__ T L[kPackMax];
  const int h = blockIdx.x, side = G + 1, P = side * (side + 1) / 2;
  const T* src = factor + (per_head ? (size_t)h * P : 0);
  for (int x = threadIdx.x; x < P; x += kThreads) L[x] = src[x];
  __syncthreads();
  for (int x = threadIdx.x; x < side * side; x += kThreads) {
    const int i = x / side, j = x % side, n = i < j ? i : j;
    double acc = 0;
    for (int m = 0; m <= n; ++m) acc += (double)L[packed(i, m)] * L[packed(j, m)];
    if (x == 0)
      c0[h] = (T)(acc + eps);
    else if (i == 0)
      lam[(size_t)h * G + j - 1] = (T)(2 * acc);
    else if (j > 0)
      gam[((size_t)h * G + i - 1) * G + j - 1] = (T)acc;
  }
}

// dL_im = sum_{j >= m} S_ij L_jm with S = dM + dM^T, a shared factor's S being the
// sum over the heads: its L is the same for all of them, so the product is formed
// once. With per_head a block takes a head's whole factor; a shared factor has a
// block for each row i, whose threads share the heads of the row's entries out and
// add them up in a fixed order. Expansion and VJP of 64 heads of 64 groups, with the
// host: 52 us; 3725 with all heads' products in one block, 437 as torch operations (256
// heads of 22 groups 53, 1356, 356). Any of dc0, dlam, dgam may be null. Sums in fp64.
template <typename T>
__global__ __launch_bounds__(kThreads) void k_expand_factor_bwd(const T* __restrict__ factor, bool per_head, int Hq,
                                                                int G, const T* __restrict__ dc0,
                                                                const T* __restrict__ dlam,
                                                                const T* __restrict__ dgam, T* __restrict__ dfactor) {
  __shared__ T L[kPackMax];
  __shared__ double S[kSideMax * kSideMax];
  static_assert(kSideMax * kSideMax >= kThreads, "the heads' parts of one row fit");
  const int side = G + 1, P = side * (side + 1) / 2;
  const int first = per_head ? blockIdx.x : 0, heads = per_head ? 1 : Hq;
  const int row0 = per_head ? 0 : blockIdx.x, rows = per_head ? side : 1;
  for (int x = threadIdx.x; x < P; x += kThreads) L[x] = factor[(size_t)first * P + x];
  const int n = rows * side, parts = max(1, min(heads, kThreads / n));
  for (int y = threadIdx.x; y < n * parts; y += kThreads) {
    const int i = row0 + y % n / side, j = y % side;
    double s = 0;
#pragma unroll 4
    for (int e = y / n; e < heads; e += parts) {
      const size_t h = first + e;
      if (i == 0 && j == 0)
        s += dc0 ? 2 * (double)dc0[h] : 0.0;
      else if (i == 0 || j == 0)
        s += dlam ? 2 * (double)dlam[h * G + i + j - 1] : 0.0;
      else if (dgam)
        s += (double)dgam[(h * G + i - 1) * G + j - 1] + dgam[(h * G + j - 1) * G + i - 1];
    }
    S[y] = s;
  }
  __syncthreads();
  if (parts > 1) {
    if (threadIdx.x < n)
      for (int p = 1; p < parts; ++p) S[threadIdx.x] += S[p * n + threadIdx.x];
    __syncthreads();
  }
  const int begin = packed(row0, 0), count = packed(row0 + rows, 0) - begin;
  for (int x = threadIdx.x; x < count; x += kThreads) {
    int i = row0;
    while (packed(i + 1, 0) <= begin + x) ++i;
    const int m = begin + x - packed(i, 0);
    double acc = 0;
    for (int j = m; j < side; ++j) acc += S[(i - row0) * side + j] * L[packed(j, m)];
    dfactor[(size_t)first * P + begin + x] = (T)acc;
  }
}

// One block per query head; dimensions past D are zero.
__global__ __launch_bounds__(kThreads) void k_expand_pairs(const float* __restrict__ b, const float* __restrict__ c,
                                                           int D, float* __restrict__ lam, float* __restrict__ gam,
                                                           int32_t* __restrict__ labels) {
  const int h = blockIdx.x, P = D * (D + 1) / 2;
  for (int x = threadIdx.x; x < kD * kD; x += kThreads) {
    const int i = x / kD, j = x % kD, hi = i > j ? i : j, lo = i > j ? j : i;
    gam[(size_t)h * kD * kD + x] = hi < D ? c[(size_t)h * P + packed(hi, lo)] : 0.f;
  }
  if (threadIdx.x < kD) {
    const int d = threadIdx.x;
    lam[h * kD + d] = d < D ? b[h * D + d] : 0.f;
    labels[h * kD + d] = d;
  }
}
__global__ __launch_bounds__(kThreads) void k_expand_pairs_bwd(const float* __restrict__ dgam, int D,
                                                               float* __restrict__ dc) {
  const int h = blockIdx.x, P = D * (D + 1) / 2;
  const float* g = dgam + (size_t)h * kD * kD;
  for (int x = threadIdx.x; x < kD * kD; x += kThreads) {
    const int i = x / kD, j = x % kD;
    if (i < D && j <= i) dc[(size_t)h * P + packed(i, j)] = i == j ? g[x] : g[x] + g[j * kD + i];
  }
}

// One wave per label row (one row shared by all heads, or one per head): ids in
// [0, G) forming a prefix. flag |= 1: an id out of range, |= 2: not a prefix.
template <typename I>
__global__ __launch_bounds__(64) void k_check_labels(const I* __restrict__ labels, bool per_head, int D, int Hq, int G,
                                                     int32_t* __restrict__ table, int* flag) {
  const int row = blockIdx.x, l = threadIdx.x;
  const I id = l < D ? labels[(size_t)row * D + l] : 0;
  const bool in = id >= 0 && id < (I)G;
  uint64_t used = l < D && in && id < 64 ? 1ull << id : 0;
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) used |= __shfl_xor(used, off, 64);
  const bool wild = __any(l < D && !in), far = __any(l < D && in && id >= 64);
  if (l == 0 && (wild || far || (used & (used + 1)) || !used)) atomicOr_system(flag, wild ? 1 : 2);
  const int32_t v = l < D && in ? (int32_t)id : 0;
  if (per_head) {
    table[(size_t)row * kD + l] = v;
  } else {
    for (int h = 0; h < Hq; ++h) table[(size_t)h * kD + l] = v;
  }
}

namespace {

__device__ __forceinline__ bool finite(float x) { return (__float_as_uint(x) & 0x7f800000u) != 0x7f800000u; }
__device__ __forceinline__ bool finite(double x) {
  return ((uint64_t)__double_as_longlong(x) & 0x7ff0000000000000ull) != 0x7ff0000000000000ull;
}
struct Bf16 {
  uint16_t x;
};
struct Fp16 {
  uint16_t x;
};
__device__ __forceinline__ bool finite(Bf16 v) { return (v.x & 0x7f80) != 0x7f80; }
__device__ __forceinline__ bool finite(Fp16 v) { return (v.x & 0x7c00) != 0x7c00; }

// Whether a thread's share of rows x width values (row stride in elements) is
// finite; 16 bytes at a time where the rows are contiguous and aligned.
template <typename T>
__device__ __forceinline__ bool all_finite(const T* __restrict__ p, size_t rows, int width, int stride, size_t t,
                                           size_t n) {
  constexpr int V = 16 / sizeof(T);
  const size_t total = rows * width;
  bool ok = true;
  size_t done = 0;
  if (stride == width && (reinterpret_cast<uintptr_t>(p) & 15) == 0) {
    struct alignas(16) Vec {
      T v[V];
    };
    const size_t vecs = total / V;
#pragma unroll 4
    for (size_t i = t; i < vecs; i += n) {
      const Vec x = reinterpret_cast<const Vec*>(p)[i];
#pragma unroll
      for (int e = 0; e < V; ++e) ok &= finite(x.v[e]);
    }
    done = vecs * V;
  }
  for (size_t i = done + t; i < total; i += n) ok &= finite(p[i / width * stride + i % width]);
  return ok;
}

}  // namespace

// flag |= 1: num or den not finite, |= 2: den not positive, |= 4: out not
// finite. num and out may be null.
template <typename T, typename O>
__global__ __launch_bounds__(kThreads) void k_check_outputs(const T* __restrict__ num, const T* __restrict__ den,
                                                            const O* __restrict__ out, size_t rows, int width,
                                                            int num_stride, int out_stride, int* flag) {
  const size_t t = (size_t)blockIdx.x * kThreads + threadIdx.x, n = (size_t)gridDim.x * kThreads;
  int bad = 0;
  for (size_t i = t; i < rows; i += n) {
    const T z = den[i];
    bad |= (finite(z) ? 0 : 1) | (z > 0 ? 0 : 2);
  }
  if (num && !all_finite(num, rows, width, num_stride, t, n)) bad |= 1;
  if (out && !all_finite(out, rows, width, out_stride, t, n)) bad |= 4;
  const int any = (__any(bad & 1) ? 1 : 0) | (__any(bad & 2) ? 2 : 0) | (__any(bad & 4) ? 4 : 0);
  if (any && (threadIdx.x & 63) == 0) atomicOr_system(flag, any);
}

namespace {

// 8 consecutive values as floats.
__device__ __forceinline__ void load8(float (&x)[8], const float* p) {
  const float4 a = reinterpret_cast<const float4*>(p)[0], b = reinterpret_cast<const float4*>(p)[1];
  x[0] = a.x, x[1] = a.y, x[2] = a.z, x[3] = a.w, x[4] = b.x, x[5] = b.y, x[6] = b.z, x[7] = b.w;
}
__device__ __forceinline__ void load8(float (&x)[8], const uint16_t* p) {
  const uint4 a = *reinterpret_cast<const uint4*>(p);
  const uint32_t w[4] = {a.x, a.y, a.z, a.w};
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    x[2 * e] = __uint_as_float(w[e] << 16);
    x[2 * e + 1] = __uint_as_float(w[e] & 0xffff0000u);
  }
}
__device__ __forceinline__ void store8(float* p, const float (&x)[8]) {
  reinterpret_cast<float4*>(p)[0] = make_float4(x[0], x[1], x[2], x[3]);
  reinterpret_cast<float4*>(p)[1] = make_float4(x[4], x[5], x[6], x[7]);
}
__device__ __forceinline__ void store8(uint16_t* p, const float (&x)[8]) {
  uint32_t w[4];
#pragma unroll
  for (int e = 0; e < 4; ++e) w[e] = from_f<uint16_t>(x[2 * e]) | (uint32_t)from_f<uint16_t>(x[2 * e + 1]) << 16;
  *reinterpret_cast<uint4*>(p) = make_uint4(w[0], w[1], w[2], w[3]);
}

}  // namespace

// One thread: 8 dimensions d .. of a head's lower half and their partners d + 32.
// back: head-first gradients -> projection gradients (the transposed rotation).
// Null tensors are skipped. Arithmetic in fp32, one rounding to T.
template <typename T, bool BACK>
__global__ __launch_bounds__(kThreads) void k_rotary_heads(T* __restrict__ pq, T* __restrict__ pk, T* __restrict__ pv,
                                                           T* __restrict__ hq, T* __restrict__ hk, T* __restrict__ hv,
                                                           const T* __restrict__ cosine, const T* __restrict__ sine,
                                                           int B, int N, int Hq, int Hkv) {
  constexpr int kHalf = kD / 2, kOct = kHalf / 8;
  const size_t x = (size_t)blockIdx.x * kThreads + threadIdx.x;
  const int heads = Hq + 2 * Hkv;
  if (x >= (size_t)B * N * heads * kOct) return;
  const int d = 8 * (int)(x % kOct);
  const int hh = (int)(x / kOct % heads);
  const size_t row = x / kOct / heads;  // b N + n
  const int n = (int)(row % N);
  const size_t b = row / N;
  const bool is_q = hh < Hq, is_v = hh >= Hq + Hkv;
  T* const proj = is_q ? pq : is_v ? pv : pk;
  T* const head = is_q ? hq : is_v ? hv : hk;
  if (!proj || !head) return;
  const int H = is_q ? Hq : Hkv, h = is_q ? hh : is_v ? hh - Hq - Hkv : hh - Hq;
  T* const p = proj + (row * H + h) * kD + d;
  T* const y = head + ((b * H + h) * N + n) * kD + d;
  float lo[8], hi[8];
  load8(lo, BACK ? y : p);
  load8(hi, (BACK ? y : p) + kHalf);
  if (!is_v) {
    float cl[8], ch[8], sl[8], sh[8];
    load8(cl, cosine + (size_t)n * kD + d);
    load8(ch, cosine + (size_t)n * kD + d + kHalf);
    load8(sl, sine + (size_t)n * kD + d);
    load8(sh, sine + (size_t)n * kD + d + kHalf);
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const float a = lo[e], c = hi[e];
      lo[e] = BACK ? a * cl[e] + c * sh[e] : a * cl[e] - c * sl[e];
      hi[e] = BACK ? c * ch[e] - a * sl[e] : c * ch[e] + a * sh[e];
    }
  }
  store8(BACK ? p : y, lo);
  store8((BACK ? p : y) + kHalf, hi);
}

template <typename T>
void launch_expand_factor(const T* factor, bool per_head, int Hq, int G, double eps, T* c0, T* lam, T* gam,
                          hipStream_t st) {
  hipLaunchKernelGGL(k_expand_factor<T>, dim3(Hq), dim3(kThreads), 0, st, factor, per_head, G, (T)eps, c0, lam, gam);
}
template <typename T>
void launch_expand_factor_bwd(const T* factor, bool per_head, int Hq, int G, const T* dc0, const T* dlam,
                              const T* dgam, T* dfactor, hipStream_t st) {
  hipLaunchKernelGGL(k_expand_factor_bwd<T>, dim3(per_head ? Hq : G + 1), dim3(kThreads), 0, st, factor, per_head, Hq,
                     G, dc0, dlam, dgam, dfactor);
}
template void launch_expand_factor<float>(const float*, bool, int, int, double, float*, float*, float*, hipStream_t);
template void launch_expand_factor<double>(const double*, bool, int, int, double, double*, double*, double*, hipStream_t);
template void launch_expand_factor_bwd<float>(const float*, bool, int, int, const float*, const float*, const float*,
                                              float*, hipStream_t);
template void launch_expand_factor_bwd<double>(const double*, bool, int, int, const double*, const double*,
                                               const double*, double*, hipStream_t);

void launch_expand_pairs(const float* b, const float* c, int Hq, int D, float* lam, float* gam, int32_t* labels,
                         hipStream_t st) {
  hipLaunchKernelGGL(k_expand_pairs, dim3(Hq), dim3(kThreads), 0, st, b, c, D, lam, gam, labels);
}
void launch_expand_pairs_bwd(const float* dgam, int Hq, int D, float* dc, hipStream_t st) {
  hipLaunchKernelGGL(k_expand_pairs_bwd, dim3(Hq), dim3(kThreads), 0, st, dgam, D, dc);
}

void launch_rotary_heads(bool f32, bool back, void* const (&t)[6], const void* cosine, const void* sine, int B, int N,
                         int Hq, int Hkv, hipStream_t st) {
  const size_t threads = (size_t)B * N * (Hq + 2 * Hkv) * (kD / 16);
  const dim3 grid((unsigned)((threads + kThreads - 1) / kThreads)), block(kThreads);
  auto launch = [&](auto* kernel, auto zero) {
    using T = decltype(zero);
    hipLaunchKernelGGL(kernel, grid, block, 0, st, static_cast<T*>(t[0]), static_cast<T*>(t[1]), static_cast<T*>(t[2]),
                       static_cast<T*>(t[3]), static_cast<T*>(t[4]), static_cast<T*>(t[5]),
                       static_cast<const T*>(cosine), static_cast<const T*>(sine), B, N, Hq, Hkv);
  };
  if (f32)
    back ? launch(k_rotary_heads<float, true>, 0.f) : launch(k_rotary_heads<float, false>, 0.f);
  else
    back ? launch(k_rotary_heads<uint16_t, true>, uint16_t{}) : launch(k_rotary_heads<uint16_t, false>, uint16_t{});
}

void launch_check_labels(const void* labels, bool wide, bool per_head, int D, int Hq, int G, int32_t* table, int* flag,
                         hipStream_t st) {
  const dim3 grid(per_head ? Hq : 1), block(64);
  if (wide)
    hipLaunchKernelGGL(k_check_labels<int64_t>, grid, block, 0, st, static_cast<const int64_t*>(labels), per_head, D, Hq,
                       G, table, flag);
  else
    hipLaunchKernelGGL(k_check_labels<int32_t>, grid, block, 0, st, static_cast<const int32_t*>(labels), per_head, D, Hq,
                       G, table, flag);
}

namespace {
template <typename T, typename O>
void check_outputs(const void* num, const void* den, const void* out, size_t rows, int width, int ns, int os, int* flag,
                   hipStream_t st) {
  // one pass at memory speed for large outputs, one block for a few rows
  const size_t work = num || out ? rows * width / 16 : rows / 4;
  const unsigned blocks = (unsigned)std::min<size_t>(2048, std::max<size_t>(1, (work + kThreads - 1) / kThreads));
  hipLaunchKernelGGL((k_check_outputs<T, O>), dim3(blocks), dim3(kThreads), 0, st, static_cast<const T*>(num),
                     static_cast<const T*>(den), static_cast<const O*>(out), rows, width, ns, os, flag);
}
}  // namespace

// out_kind: 0 float32, 1 bfloat16, 2 float16, 3 float64.
int launch_check_outputs(bool wide, int out_kind, const void* num, const void* den, const void* out, size_t rows,
                         int width, int num_stride, int out_stride, int* flag, hipStream_t st) {
#define OAL_CHECK(T, O) check_outputs<T, O>(num, den, out, rows, width, num_stride, out_stride, flag, st)
  switch (out_kind + (wide ? 4 : 0)) {
    case 0: OAL_CHECK(float, float); break;
    case 1: OAL_CHECK(float, Bf16); break;
    case 2: OAL_CHECK(float, Fp16); break;
    case 3: OAL_CHECK(float, double); break;
    case 4: OAL_CHECK(double, float); break;
    case 5: OAL_CHECK(double, Bf16); break;
    case 6: OAL_CHECK(double, Fp16); break;
    case 7: OAL_CHECK(double, double); break;
    default: return 1;
  }
#undef OAL_CHECK
  return 0;
}

}  // namespace oal
