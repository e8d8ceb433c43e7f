// FP64 evaluation of the grouped quadratic operator for gfx950: the HIP route
// of oal_attention(execution="reference") when the working dtype is float64.
//
// The reference evaluates that execution in the working dtype
// (oal_attention/grouped_quadratic.py:332-355, grouped_reference.py:102-211),
// and its gradients come from torch autograd of that evaluation. Here the
// operator is evaluated over token pairs, every operand and every sum in fp64:
//   p_d(i,j) = scale q_i[d] k_j[d]              (d < 64)
//   kappa    = c0 + sum_d a_d p_d + sum_{d,e} A_de p_d p_e
//   a_d      = lam[g(d)],  A_de = gam[g(d)][g(e)]
// which is the reference's kappa (s_g = sum_{d in g} p_d). Per pair, with
// inner_d = sum_e A_de p_e:
//   kappa = c0 + sum_d p_d (a_d + inner_d),   d kappa / d p_d = a_d + 2 inner_d.
// num_i = sum_{j<=i} kappa_ij v_j, den_i = sum_{j<=i} kappa_ij, out = num / den.
// VJP (normalization as hd_block_gemm_normalization_ops.py:32-71 without a floor):
//   G_i = dout_i / den_i + dnum_i,  Gz_i = -(dout_i . num_i) / den_i^2 + dden_i
//   ds_ij = G_i . v_j + Gz_i
//   dq_i[d] += ds_ij scale k_j[d] (a_d + 2 inner_d),  dk_j[d] likewise with q_i[d]
//   dv_j += kappa_ij G_i
//   dW[f] = sum ds_ij p_r p_c over the feature (r, c) table (p_64 = 1), routed to
//   dc0 = dW[0], dlam[g] = sum_{d in g} dW[1 + d],
//   dgam[g][h] = sum_{d in g, e in h} dW[pair(max(d,e), min(d,e))]
// (dgam is d/dgam of sum_{g,h} gam_gh s_g s_h, the convention of the fp32 and
// bf16 routes; a factor's gradient is the same under the reference's gather).
//
// Up to 8 groups (kGroups) the pair values come from group sums on the fp64
// matrix cores (the k64g_* kernels below): O(N^2 (64 + G^2)) per head. More
// groups take the per-dimension kernels (k64_*): 64 * 64 terms a pair whatever the
// labels, tiles of 32 queries x 32 keys, a block's 128 threads being 32 tokens x
// 4 quarters, each quarter owning 16 of the 64 dimensions. Kernel time of one
// forward and backward at B=1, Hq=14, Hkv=2, N=256 and 8 groups: 43.4 ms from
// per-dimension sums (32.8 in k64_dkv's 16 blocks), 0.17 ms from group sums
// (k64g_fwd 30, k64g_dq 67, k64g_dkv 53 us; at N=1024 160, 400 and 361 us).

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "oal_common.hpp"
#include "oal_internal.hpp"
#include "oal_layout.hpp"

namespace oal {

static __constant__ FeatureTable kTab64 = make_feature_table();

namespace {

constexpr int kT = 32;         // tokens per tile
constexpr int kS = kD + 2;     // LDS row stride in doubles (16-byte aligned rows)
constexpr int kNT = 4 * kT;    // threads per block
constexpr int kCoefThreads = 256;
constexpr int kCoefSlots = (kFeat + kCoefThreads - 1) / kCoefThreads;  // features per thread

// Rows [tok0, tok0 + kT) of a [N][64] fp64 matrix into LDS; rows past N are zero.
__device__ __forceinline__ void stage_tile(double (*dst)[kS], const double* __restrict__ src, int tok0, int N) {
  for (int idx = threadIdx.x; idx < kT * (kD / 2); idx += blockDim.x) {
    const int r = idx / (kD / 2), c2 = idx % (kD / 2), tok = tok0 + r;
    double2 x = make_double2(0.0, 0.0);
    if (tok < N) x = reinterpret_cast<const double2*>(src + (size_t)tok * kD)[c2];
    reinterpret_cast<double2*>(&dst[r][0])[c2] = x;
  }
}

// G and Gz rows of a query tile: [G_i (64), Gz_i] per row; rows past N are zero.
__device__ __forceinline__ void stage_grad_tile(double (*dst)[kS], const double* __restrict__ Gv,
                                                const double* __restrict__ Gz, int tok0, int N) {
  stage_tile(dst, Gv, tok0, N);
  for (int r = threadIdx.x; r < kT; r += blockDim.x) dst[r][kD] = tok0 + r < N ? Gz[tok0 + r] : 0.0;
}

// Per-dimension coefficients of head h: A[d][e] = gam[g(d)][g(e)], A[d][64] =
// lam[g(d)]. Labels are clamped into [0, G) (the host validates them).
__device__ void stage_coefficients(double (*A)[kS], int* lab, const int32_t* __restrict__ labels,
                                   const double* __restrict__ lam, const double* __restrict__ gam, int G, int h) {
  __syncthreads();
  if (threadIdx.x < kD) {
    const int g = labels[h * kD + threadIdx.x];
    lab[threadIdx.x] = g < 0 ? 0 : (g >= G ? G - 1 : g);
  }
  __syncthreads();
  for (int idx = threadIdx.x; idx < kD * (kD + 1); idx += blockDim.x) {
    const int d = idx / (kD + 1), e = idx % (kD + 1);
    A[d][e] = e < kD ? gam[((size_t)h * G + lab[d]) * G + lab[e]] : lam[(size_t)h * G + lab[d]];
  }
  __syncthreads();
}

// Sum over the four quarters of a token (lanes 4 t .. 4 t + 3).
__device__ __forceinline__ double quarter_sum(double x) {
  x += __shfl_xor(x, 1, 64);
  x += __shfl_xor(x, 2, 64);
  return x;
}

// The quarter's part of a pair's p vector: pm[m] = scale x[d] y[d] for
// d = 16 cq + m, also written to the token's LDS row prow (the four quarters of
// a token are lanes of one wave, whose LDS accesses complete in program order,
// so the row is whole when the quarters read it back).
__device__ __forceinline__ void quarter_products(const double* x, const double* y, double scale, int cq,
                                                 double* prow, double (&pm)[16]) {
#pragma unroll
  for (int m = 0; m < 16; m += 2) {
    const int d = 16 * cq + m;
    const double2 a = *reinterpret_cast<const double2*>(x + d);
    const double2 b = *reinterpret_cast<const double2*>(y + d);
    pm[m] = scale * a.x * b.x;
    pm[m + 1] = scale * a.y * b.y;
    *reinterpret_cast<double2*>(prow + d) = make_double2(pm[m], pm[m + 1]);
  }
}

// inner_d = sum_e A[d][e] p[e] for the quarter's 16 dimensions d = 16 cq + m,
// p read back from the token's LDS row.
__device__ __forceinline__ void quarter_inner(const double (*A)[kS], int cq, const double* prow,
                                              double (&inner)[16]) {
#pragma unroll
  for (int m = 0; m < 16; ++m) inner[m] = 0.0;
#pragma unroll 2
  for (int e = 0; e < kD; e += 2) {
    const double2 pe = *reinterpret_cast<const double2*>(prow + e);
#pragma unroll
    for (int m = 0; m < 16; ++m) {
      const double2 w = *reinterpret_cast<const double2*>(&A[16 * cq + m][e]);
      inner[m] = fma(w.y, pe.y, fma(w.x, pe.x, inner[m]));
    }
  }
}

}  // namespace

// ---------------------------------------------------------------------------
// Forward: one block per (query tile, batch x query head).
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(kNT) void k64_fwd(const double* __restrict__ q, const double* __restrict__ k,
                                               const double* __restrict__ v, const int32_t* __restrict__ labels,
                                               const double* __restrict__ c0, const double* __restrict__ lam,
                                               const double* __restrict__ gam, int G, int Hq, int Hkv, int N,
                                               double scale, double* __restrict__ out, double* __restrict__ num,
                                               double* __restrict__ den) {
  __shared__ __attribute__((aligned(16))) double A[kD][kS];
  __shared__ __attribute__((aligned(16))) double qs[kT][kS];
  __shared__ __attribute__((aligned(16))) double ks[kT][kS];
  __shared__ __attribute__((aligned(16))) double vs[kT][kS];
  __shared__ __attribute__((aligned(16))) double ps[kT][kS];  // p of each token's current pair
  __shared__ int lab[kD];
  const int it = blockIdx.x, bh = blockIdx.y;
  const int b = bh / Hq, h = bh % Hq, u = b * Hkv + h / (Hq / Hkv);
  const int t = threadIdx.x, i = t >> 2, cq = t & 3;
  const int tq = it * kT + i;
  stage_coefficients(A, lab, labels, lam, gam, G, h);
  stage_tile(qs, q + (size_t)bh * N * kD, it * kT, N);
  const double cc = c0[h];
  double acc[16];
#pragma unroll
  for (int m = 0; m < 16; ++m) acc[m] = 0.0;
  double accz = 0.0;
  for (int jt = 0; jt <= it; ++jt) {
    __syncthreads();
    stage_tile(ks, k + (size_t)u * N * kD, jt * kT, N);
    stage_tile(vs, v + (size_t)u * N * kD, jt * kT, N);
    __syncthreads();
    for (int j = 0; j < kT; ++j) {
      double pm[16], inner[16];
      quarter_products(qs[i], ks[j], scale, cq, ps[i], pm);
      quarter_inner(A, cq, ps[i], inner);
      double part = 0.0;
#pragma unroll
      for (int m = 0; m < 16; ++m) part = fma(pm[m], A[16 * cq + m][kD] + inner[m], part);
      part = quarter_sum(part);
      const int tk = jt * kT + j;
      const double kap = (tk <= tq && tk < N) ? cc + part : 0.0;
#pragma unroll
      for (int m = 0; m < 16; ++m) acc[m] = fma(kap, vs[j][16 * cq + m], acc[m]);
      accz += kap;
    }
  }
  if (tq < N) {
    const size_t o = ((size_t)bh * N + tq) * kD + 16 * cq;
#pragma unroll
    for (int m = 0; m < 16; ++m) {
      num[o + m] = acc[m];
      out[o + m] = acc[m] / accz;
    }
    if (cq == 0) den[(size_t)bh * N + tq] = accz;
  }
}

// ---------------------------------------------------------------------------
// Normalization VJP, one wave per row.
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(256) void k64_gvec(const double* __restrict__ dout, const double* __restrict__ dnum,
                                                const double* __restrict__ dden, const double* __restrict__ num,
                                                const double* __restrict__ den, long rows, double* __restrict__ Gv,
                                                double* __restrict__ Gz) {
  const long row = (long)blockIdx.x * 4 + (threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  if (row >= rows) return;
  const double dd = den[row];
  const double dO = dout ? dout[row * kD + lane] : 0.0;
  double g = dO / dd;
  if (dnum) g += dnum[row * kD + lane];
  Gv[row * kD + lane] = g;
  double dot = dO * num[row * kD + lane];
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) dot += __shfl_xor(dot, off, 64);
  if (lane == 0) {
    double gz = -dot / (dd * dd);
    if (dden) gz += dden[row];
    Gz[row] = gz;
  }
}

// ---------------------------------------------------------------------------
// Query-side VJP: one block per (query tile, batch x query head).
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(kNT) void k64_dq(const double* __restrict__ q, const double* __restrict__ k,
                                              const double* __restrict__ v, const int32_t* __restrict__ labels,
                                              const double* __restrict__ lam, const double* __restrict__ gam, int G,
                                              int Hq, int Hkv, int N, double scale, const double* __restrict__ Gv,
                                              const double* __restrict__ Gz, double* __restrict__ dq) {
  __shared__ __attribute__((aligned(16))) double A[kD][kS];
  __shared__ __attribute__((aligned(16))) double qs[kT][kS];
  __shared__ __attribute__((aligned(16))) double gs[kT][kS];
  __shared__ __attribute__((aligned(16))) double ks[kT][kS];
  __shared__ __attribute__((aligned(16))) double vs[kT][kS];
  __shared__ __attribute__((aligned(16))) double ps[kT][kS];  // p of each token's current pair
  __shared__ int lab[kD];
  const int it = blockIdx.x, bh = blockIdx.y;
  const int b = bh / Hq, h = bh % Hq, u = b * Hkv + h / (Hq / Hkv);
  const int t = threadIdx.x, i = t >> 2, cq = t & 3;
  const int tq = it * kT + i;
  stage_coefficients(A, lab, labels, lam, gam, G, h);
  stage_tile(qs, q + (size_t)bh * N * kD, it * kT, N);
  stage_grad_tile(gs, Gv + (size_t)bh * N * kD, Gz + (size_t)bh * N, it * kT, N);
  double acc[16];
#pragma unroll
  for (int m = 0; m < 16; ++m) acc[m] = 0.0;
  for (int jt = 0; jt <= it; ++jt) {
    __syncthreads();
    stage_tile(ks, k + (size_t)u * N * kD, jt * kT, N);
    stage_tile(vs, v + (size_t)u * N * kD, jt * kT, N);
    __syncthreads();
    for (int j = 0; j < kT; ++j) {
      double ds = 0.0;
#pragma unroll
      for (int m = 0; m < 16; ++m) ds = fma(gs[i][16 * cq + m], vs[j][16 * cq + m], ds);
      ds = quarter_sum(ds) + gs[i][kD];
      const int tk = jt * kT + j;
      if (!(tk <= tq && tk < N)) ds = 0.0;
      double pm[16], inner[16];
      quarter_products(qs[i], ks[j], scale, cq, ps[i], pm);
      quarter_inner(A, cq, ps[i], inner);
      const double sds = ds * scale;
#pragma unroll
      for (int m = 0; m < 16; ++m) {
        const int d = 16 * cq + m;
        acc[m] = fma(sds * ks[j][d], A[d][kD] + 2.0 * inner[m], acc[m]);
      }
    }
  }
  if (tq < N) {
    const size_t o = ((size_t)bh * N + tq) * kD + 16 * cq;
#pragma unroll
    for (int m = 0; m < 16; ++m) dq[o + m] = acc[m];
  }
}

// ---------------------------------------------------------------------------
// Key/value-side VJP: one block per (key tile, unit = batch x KV head), summed
// over the unit's query heads in head order.
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(kNT) void k64_dkv(const double* __restrict__ q, const double* __restrict__ k,
                                               const double* __restrict__ v, const int32_t* __restrict__ labels,
                                               const double* __restrict__ c0, const double* __restrict__ lam,
                                               const double* __restrict__ gam, int G, int Hq, int Hkv, int N,
                                               double scale, const double* __restrict__ Gv,
                                               const double* __restrict__ Gz, double* __restrict__ dk,
                                               double* __restrict__ dv) {
  __shared__ __attribute__((aligned(16))) double A[kD][kS];
  __shared__ __attribute__((aligned(16))) double qs[kT][kS];
  __shared__ __attribute__((aligned(16))) double gs[kT][kS];
  __shared__ __attribute__((aligned(16))) double ks[kT][kS];
  __shared__ __attribute__((aligned(16))) double vs[kT][kS];
  __shared__ __attribute__((aligned(16))) double ps[kT][kS];  // p of each token's current pair
  __shared__ int lab[kD];
  const int jt = blockIdx.x, u = blockIdx.y;
  const int R = Hq / Hkv, b = u / Hkv, kh = u % Hkv;
  const int NT = (N + kT - 1) / kT;
  const int t = threadIdx.x, j = t >> 2, cq = t & 3;
  const int tk = jt * kT + j;
  stage_tile(ks, k + (size_t)u * N * kD, jt * kT, N);
  stage_tile(vs, v + (size_t)u * N * kD, jt * kT, N);
  double dka[16], dva[16];
#pragma unroll
  for (int m = 0; m < 16; ++m) dka[m] = dva[m] = 0.0;
  for (int hh = 0; hh < R; ++hh) {
    const int h = kh * R + hh, bh = b * Hq + h;
    stage_coefficients(A, lab, labels, lam, gam, G, h);
    const double cc = c0[h];
    for (int it = jt; it < NT; ++it) {
      __syncthreads();
      stage_tile(qs, q + (size_t)bh * N * kD, it * kT, N);
      stage_grad_tile(gs, Gv + (size_t)bh * N * kD, Gz + (size_t)bh * N, it * kT, N);
      __syncthreads();
      for (int i = 0; i < kT; ++i) {
        const int tq = it * kT + i;
        const bool ok = tk <= tq && tq < N && tk < N;
        double pm[16], inner[16];
        quarter_products(qs[i], ks[j], scale, cq, ps[j], pm);
        quarter_inner(A, cq, ps[j], inner);
        double part = 0.0, ds = 0.0;
#pragma unroll
        for (int m = 0; m < 16; ++m) {
          const int d = 16 * cq + m;
          part = fma(pm[m], A[d][kD] + inner[m], part);
          ds = fma(gs[i][d], vs[j][d], ds);
        }
        part = quarter_sum(part);
        ds = quarter_sum(ds) + gs[i][kD];
        const double kap = ok ? cc + part : 0.0;
        const double sds = ok ? ds * scale : 0.0;
#pragma unroll
        for (int m = 0; m < 16; ++m) {
          const int d = 16 * cq + m;
          dva[m] = fma(kap, gs[i][d], dva[m]);
          dka[m] = fma(sds * qs[i][d], A[d][kD] + 2.0 * inner[m], dka[m]);
        }
      }
    }
  }
  if (tk < N) {
    const size_t o = ((size_t)u * N + tk) * kD + 16 * cq;
#pragma unroll
    for (int m = 0; m < 16; ++m) {
      if (dk) dk[o + m] = dka[m];
      if (dv) dv[o + m] = dva[m];
    }
  }
}

// ---------------------------------------------------------------------------
// Coefficient partials: one block per (query tile, batch x query head);
// part[bh][it][f] = sum over the tile's pairs of ds p_r p_c for feature f =
// (r, c) of the feature table (p_64 = 1, padding features 0). Each thread owns
// features f = t + 256 m; a query row's 32 pairs are staged at a time.
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(kCoefThreads) void k64_coef_part(const double* __restrict__ q,
                                                              const double* __restrict__ k,
                                                              const double* __restrict__ v, int Hq, int Hkv, int N,
                                                              double scale, const double* __restrict__ Gv,
                                                              const double* __restrict__ Gz,
                                                              double* __restrict__ part) {
  __shared__ __attribute__((aligned(16))) double qs[kT][kS];
  __shared__ __attribute__((aligned(16))) double gs[kT][kS];
  __shared__ __attribute__((aligned(16))) double ks[kT][kS];
  __shared__ __attribute__((aligned(16))) double vs[kT][kS];
  __shared__ __attribute__((aligned(16))) double pr[kT][kS];  // p of one query row: [key][64 dims, 1, 0]
  __shared__ double dsr[kT];
  const int it = blockIdx.x, bh = blockIdx.y;
  const int NT = (N + kT - 1) / kT;
  const int b = bh / Hq, h = bh % Hq, u = b * Hkv + h / (Hq / Hkv);
  const int t = threadIdx.x;
  int fr[kCoefSlots], fc[kCoefSlots];
  double acc[kCoefSlots];
#pragma unroll
  for (int m = 0; m < kCoefSlots; ++m) {
    const int f = t + kCoefThreads * m;
    fr[m] = f < kFeat ? kTab64.r[f] : kD + 1;
    fc[m] = f < kFeat ? kTab64.c[f] : kD + 1;
    acc[m] = 0.0;
  }
  stage_tile(qs, q + (size_t)bh * N * kD, it * kT, N);
  stage_grad_tile(gs, Gv + (size_t)bh * N * kD, Gz + (size_t)bh * N, it * kT, N);
  for (int r = t; r < kT; r += blockDim.x) {
    pr[r][kD] = 1.0;
    pr[r][kD + 1] = 0.0;
  }
  for (int jt = 0; jt <= it; ++jt) {
    __syncthreads();
    stage_tile(ks, k + (size_t)u * N * kD, jt * kT, N);
    stage_tile(vs, v + (size_t)u * N * kD, jt * kT, N);
    for (int i = 0; i < kT; ++i) {
      __syncthreads();
      const int tq = it * kT + i;
      for (int idx = t; idx < kT * kD; idx += blockDim.x) {
        const int jj = idx / kD, d = idx % kD;
        pr[jj][d] = scale * qs[i][d] * ks[jj][d];
      }
      if (t < kT) {
        const int tk = jt * kT + t;
        double ds = gs[i][kD];
        for (int c = 0; c < kD; ++c) ds = fma(gs[i][c], vs[t][c], ds);
        dsr[t] = (tk <= tq && tk < N && tq < N) ? ds : 0.0;
      }
      __syncthreads();
      for (int jj = 0; jj < kT; ++jj) {
        const double ds = dsr[jj];
#pragma unroll
        for (int m = 0; m < kCoefSlots; ++m) acc[m] = fma(ds * pr[jj][fr[m]], pr[jj][fc[m]], acc[m]);
      }
    }
  }
  double* dst = part + ((size_t)bh * NT + it) * kFP;
#pragma unroll
  for (int m = 0; m < kCoefSlots; ++m) {
    const int f = t + kCoefThreads * m;
    if (f < kFP) dst[f] = f < kFeat ? acc[m] : 0.0;
  }
  for (int f = t + kCoefThreads * kCoefSlots; f < kFP; f += kCoefThreads) dst[f] = 0.0;
}

// ---------------------------------------------------------------------------
// dc0, dlam, dgam of head h: the partials summed over (batch, query tile) in a
// fixed order, then routed through the labels in ascending dimension order.
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(256) void k64_coef_grad(const double* __restrict__ part, int B, int Hq, int NT,
                                                     const int32_t* __restrict__ labels, int G,
                                                     double* __restrict__ dc0, double* __restrict__ dlam,
                                                     double* __restrict__ dgam) {
  __shared__ double w[kFP];
  __shared__ int lab[kD];
  __shared__ uint8_t mem[kD][kD];  // mem[g][0 .. cnt[g]): the dimensions of group g, ascending
  __shared__ int cnt[kD];
  const int h = blockIdx.x, t = threadIdx.x;
  if (t < kD) {
    const int g = labels[h * kD + t];
    lab[t] = g < 0 ? 0 : (g >= G ? G - 1 : g);
  }
  for (int f = t; f < kFP; f += blockDim.x) {
    double acc = 0.0;
    for (int b = 0; b < B; ++b) {
      const double* src = part + ((size_t)(b * Hq + h) * NT) * kFP + f;
      for (int it = 0; it < NT; ++it) acc += src[(size_t)it * kFP];
    }
    w[f] = acc;
  }
  for (int g = t; g < G; g += blockDim.x) {
    int n = 0;
    for (int d = 0; d < kD; ++d)
      if (lab[d] == g) mem[g][n++] = (uint8_t)d;
    cnt[g] = n;
  }
  __syncthreads();
  if (t == 0) dc0[h] = w[0];
  for (int g = t; g < G; g += blockDim.x) {
    double acc = 0.0;
    for (int i = 0; i < cnt[g]; ++i) acc += w[1 + mem[g][i]];
    dlam[(size_t)h * G + g] = acc;
  }
  // every (g, h) entry walks only its two groups' members: 64 x 64 terms per
  // head in all, whatever the group count
  for (int e = t; e < G * G; e += blockDim.x) {
    const int gr = e / G, gc = e % G;
    double acc = 0.0;
    for (int i = 0; i < cnt[gr]; ++i) {
      const int d = mem[gr][i];
      for (int j = 0; j < cnt[gc]; ++j) {
        const int c = mem[gc][j];
        const int r0 = d > c ? d : c, c0i = d > c ? c : d;
        acc += w[1 + kD + r0 * (r0 + 1) / 2 + c0i];
      }
    }
    dgam[(size_t)h * G * G + e] = acc;
  }
}

// ---------------------------------------------------------------------------
// Up to kGroups groups: group sums on the matrix cores.
//
// v_mfma_f64_16x16x4_f64 runs at the rate of the fp64 VALU, so what it buys is
// operand traffic: one operand register per lane and k-step feeds 16 products,
// where the per-dimension form reads 64 x 64 coefficients from LDS for every
// pair. What bounds these kernels is fp64 issue (64 cycles a product, 4 a VALU
// instruction): about 23 products for the group sums of a 16 x 16 tile, 16 each
// for a contraction over the 64 dimensions or value columns, and 64 G-by-G FMAs
// per entry.
//
// A wave takes 16 x 16 token tiles. The dimensions are in group-sorted order
// (perm), 16 k-steps of 4, so a group is a range of positions: its sum takes the
// k-steps that its range touches, with the first operand zero outside the
// group. A tile's accumulator register r of lane l is entry
// [4 r + l / 16][l % 16], which is, as it stands, the first operand of a product
// over the tile's rows: k-step r, row l % 16 of the result. So a kernel that
// sums over keys forms the tiles transposed ([key][query]) and one that sums
// over queries forms them straight, and no tile passes through LDS.
// A block's waves share one row of tiles, taken in turn (tile index mod waves),
// and add their sums in wave order at the end: a fixed order whatever the
// device does. 14 heads of 256 tokens are 224 blocks. Eight waves, two on a SIMD,
// hide part of one another's latency and halve the longest row's chain; k64g_dq with eight
// spills 128 registers and is slower (78 against 72 us). The blocks are
// numbered with every head's longest rows first, so that the last to run are short:
// N = 1024, 14 heads, k64g_fwd 227 to 160 us, k64g_dq 571 to 400, k64g_dkv 514 to 361
// (head by head before).
// ---------------------------------------------------------------------------
namespace {

constexpr int kG64 = 8;          // groups of these kernels
constexpr int kM = 16;           // tile edge
constexpr int kWv = 8;           // waves per block
constexpr int kWvDq = 4;         // of k64g_dq: its coefficient sums take more than half of the registers
constexpr int kPairs64 = kG64 * (kG64 + 1) / 2;
constexpr int kCo = 1 + kG64 + kPairs64;  // coefficient sums: 1, s_g, s_g s_h (g >= h)

typedef double d4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ d4 mma64(double a, double b, d4 c) {
  return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}

// A head's coefficients and its dimensions in group order.
struct HeadTab {
  double c0, lam[kG64], gam[kG64][kG64];  // zero beyond the given groups
  int perm[kD], grp[kD];                  // position -> dimension, group
  int first[kG64 + 1];                    // group g holds positions [first[g], first[g + 1])
};

// Positions by ballot: one load of the labels per block. Counted label by label they
// were a chain of 64 dependent reads, twice, before the first tile.
__device__ void stage_head(HeadTab& tab, const int32_t* __restrict__ labels, const double* __restrict__ c0,
                           const double* __restrict__ lam, const double* __restrict__ gam, int G, int h) {
  const int t = threadIdx.x;
  if (t < kD) {  // the first wave: one lane per dimension
    const int own = labels[h * kD + t], g = own < 0 ? 0 : (own >= G ? G - 1 : own);
    int before = 0, pos = 0;  // dimensions of lower groups; this lane's position
#pragma unroll
    for (int e = 0; e < kG64; ++e) {
      const uint64_t members = __ballot(g == e);
      if (t == 0) tab.first[e] = before;
      if (g == e) pos = before + __popcll(members & ((1ull << t) - 1));
      before += __popcll(members);
    }
    if (t == 0) tab.first[kG64] = before;
    tab.perm[pos] = t;
    tab.grp[pos] = g;
  }
  if (t < kG64 * kG64) {
    const int a = t / kG64, b = t % kG64;
    tab.gam[a][b] = a < G && b < G ? gam[((size_t)h * G + a) * G + b] : 0.0;
  }
  if (t < kG64) tab.lam[t] = t < G ? lam[(size_t)h * G + t] : 0.0;
  if (t == 0) tab.c0 = c0 ? c0[h] : 0.0;
  __syncthreads();
}

// The wave's operand of 16 rows in group order: x[s] = row (row0 + l % 16),
// position 4 s + l / 16. Rows past N repeat row N - 1 (their entries are masked).
__device__ __forceinline__ void load_sorted(double (&x)[16], const double* __restrict__ src, int row0, int N,
                                            const HeadTab& tab, int lane) {
  const int row = row0 + (lane & 15);
  const double* p = src + (size_t)(row < N ? row : N - 1) * kD;
#pragma unroll
  for (int s = 0; s < 16; ++s) x[s] = p[tab.perm[4 * s + (lane >> 4)]];
}

// The same in the natural order of the dimensions (value columns, G).
__device__ __forceinline__ void load_rows(double (&x)[16], const double* __restrict__ src, int row0, int N, int lane) {
  const int row = row0 + (lane & 15);
  const double* p = src + (size_t)(row < N ? row : N - 1) * kD;
#pragma unroll
  for (int s = 0; s < 16; ++s) x[s] = p[4 * s + (lane >> 4)];
}

// Makes the compiler read a head's table again: kept in registers over the tile
// loop it is 144 coefficient and 256 mask registers, which spill.
__device__ __forceinline__ void reread() { asm volatile("" ::: "memory"); }

// The W-position steps that group g's range touches, one bit each. In a scalar
// register: the 128 + 32 tests of a tile are a bit test and a scalar branch each,
// and not a lane mask formed, saved and restored around every product.
template <int W>
__device__ __forceinline__ uint32_t touched(const HeadTab& tab, int g) {
  const int lo = __builtin_amdgcn_readfirstlane(tab.first[g]), hi = __builtin_amdgcn_readfirstlane(tab.first[g + 1]);
  return lo < hi ? (1u << (hi + W - 1) / W) - (1u << lo / W) : 0u;
}

// s[g] = scale * sum over the group's positions of a[row] b[col].
__device__ __forceinline__ void group_sums(d4 (&s)[kG64], const double (&a)[16], const double (&b)[16], double scale,
                                           const HeadTab& tab, int lane) {
  reread();
  int lab[16];
#pragma unroll
  for (int k = 0; k < 16; ++k) lab[k] = tab.grp[4 * k + (lane >> 4)];
#pragma unroll
  for (int g = 0; g < kG64; ++g) {
    const uint32_t steps = touched<4>(tab, g);
    d4 acc = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int k = 0; k < 16; ++k)
      if (steps >> k & 1) acc = mma64(lab[k] == g ? a[k] : 0.0, b[k], acc);
    s[g] = acc * scale;
  }
}

// t[g] = sum_h gam[g][h] s[h]
__device__ __forceinline__ d4 quadratic_row(const d4 (&s)[kG64], const HeadTab& tab, int g) {
  d4 t = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
  for (int h = 0; h < kG64; ++h) t += tab.gam[g][h] * s[h];
  return t;
}

__device__ __forceinline__ d4 kappa_tile(const d4 (&s)[kG64], const HeadTab& tab) {
  d4 kap = {tab.c0, tab.c0, tab.c0, tab.c0};
#pragma unroll
  for (int g = 0; g < kG64; ++g) kap += s[g] * (tab.lam[g] + quadratic_row(s, tab, g));
  return kap;
}

// sum over the four lane groups of a column (lanes l, l + 16, l + 32, l + 48)
__device__ __forceinline__ double column_sum(double x) {
  x += __shfl_xor(x, 16, 64);
  x += __shfl_xor(x, 32, 64);
  return x;
}

// acc[cb] += sum over the tile's rows of (ds d kappa / d s_g)[row][.] y[row][.] for the
// positions 16 cb + l % 16 of each group: the query or key gradient's products
// in group order. tile ds, operand rows y from memory; rows past N repeat row N - 1.
__device__ __forceinline__ void gradient_products(d4 (&acc)[4], const d4 (&s)[kG64], const d4& ds,
                                                  const double* __restrict__ src, int row0, int N,
                                                  const HeadTab& tab, int lane) {
  const double* rows[4];
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int row = row0 + 4 * r + (lane >> 4);
    rows[r] = src + (size_t)(row < N ? row : N - 1) * kD;
  }
  reread();
  double y[4][4];
  int lab[4];
#pragma unroll
  for (int cb = 0; cb < 4; ++cb) {
    const int pos = 16 * cb + (lane & 15), d = tab.perm[pos];
    lab[cb] = tab.grp[pos];
#pragma unroll
    for (int r = 0; r < 4; ++r) y[cb][r] = rows[r][d];
  }
#pragma unroll
  for (int g = 0; g < kG64; ++g) {
    const uint32_t blocks = touched<16>(tab, g);
    const d4 x = ds * (tab.lam[g] + 2.0 * quadratic_row(s, tab, g));
#pragma unroll
    for (int cb = 0; cb < 4; ++cb)
      if (blocks >> cb & 1) {
#pragma unroll
        for (int r = 0; r < 4; ++r) acc[cb] = mma64(x[r], lab[cb] == g ? y[cb][r] : 0.0, acc[cb]);
      }
  }
}

// acc[cb] += sum over the tile's rows of t[row][.] y[row][16 cb + l % 16].
__device__ __forceinline__ void value_products(d4 (&acc)[4], const d4& t, const double* __restrict__ src, int row0,
                                               int N, int lane) {
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int row = row0 + 4 * r + (lane >> 4);
    const double* p = src + (size_t)(row < N ? row : N - 1) * kD + (lane & 15);
#pragma unroll
    for (int cb = 0; cb < 4; ++cb) acc[cb] = mma64(t[r], p[16 * cb], acc[cb]);
  }
}

// The block's W accumulator sets summed in wave order through LDS; wave 0 holds the result.
template <int W>
__device__ __forceinline__ void add_waves(d4 (&acc)[4], double* red, int wave, int lane) {
  __syncthreads();
  if (wave) {
#pragma unroll
    for (int cb = 0; cb < 4; ++cb)
#pragma unroll
      for (int r = 0; r < 4; ++r) red[((wave - 1) * 16 + 4 * cb + r) * 64 + lane] = acc[cb][r];
  }
  __syncthreads();
  if (!wave) {
    for (int w = 0; w < W - 1; ++w)
#pragma unroll
      for (int cb = 0; cb < 4; ++cb)
#pragma unroll
        for (int r = 0; r < 4; ++r) acc[cb][r] += red[(w * 16 + 4 * cb + r) * 64 + lane];
  }
}

constexpr int red_size(int waves) { return (waves - 1) * 16 * 64; }  // doubles of add_waves' scratch

}  // namespace

__global__ __launch_bounds__(64 * kWv) void k64g_fwd(const double* __restrict__ q, const double* __restrict__ k,
                                                     const double* __restrict__ v,
                                                     const int32_t* __restrict__ labels,
                                                     const double* __restrict__ c0, const double* __restrict__ lam,
                                                     const double* __restrict__ gam, int G, int Hq, int Hkv, int N,
                                                     double scale, double* __restrict__ out,
                                                     double* __restrict__ num, double* __restrict__ den) {
  __shared__ HeadTab tab;
  __shared__ double red[red_size(kWv)];
  __shared__ double zred[kWv][kM];
  const int NT = (N + kM - 1) / kM, it = NT - 1 - (int)tile_of(blockIdx.y, blockIdx.z, gridDim.y);
  if (it < 0) return;
  const int bh = blockIdx.x, wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int b = bh / Hq, h = bh % Hq, u = b * Hkv + h / (Hq / Hkv);
  stage_head(tab, labels, c0, lam, gam, G, h);
  const int tq = it * kM + (lane & 15);
  const double* ku = k + (size_t)u * N * kD;
  const double* vu = v + (size_t)u * N * kD;
  double qr[16];
  load_sorted(qr, q + (size_t)bh * N * kD, it * kM, N, tab, lane);
  d4 acc[4] = {};
  double z = 0.0;
  for (int jt = wave; jt <= it; jt += kWv) {
    double kr[16];
    load_sorted(kr, ku, jt * kM, N, tab, lane);
    d4 s[kG64];
    group_sums(s, kr, qr, scale, tab, lane);
    d4 kap = kappa_tile(s, tab);
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int tk = jt * kM + 4 * r + (lane >> 4);
      kap[r] = tk <= tq && tk < N ? kap[r] : 0.0;
      z += kap[r];
    }
    value_products(acc, kap, vu, jt * kM, N, lane);
  }
  z = column_sum(z);
  if (lane < kM) zred[wave][lane] = z;
  add_waves<kWv>(acc, red, wave, lane);
  if (wave) return;
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int i = 4 * r + (lane >> 4), row = it * kM + i;
    if (row >= N) continue;
    double zz = 0.0;
    for (int w = 0; w < kWv; ++w) zz += zred[w][i];
    const size_t o = ((size_t)bh * N + row) * kD + (lane & 15);
#pragma unroll
    for (int cb = 0; cb < 4; ++cb) {
      num[o + 16 * cb] = acc[cb][r];
      out[o + 16 * cb] = acc[cb][r] / zz;
    }
    if ((lane & 15) == 0) den[(size_t)bh * N + row] = zz;
  }
}

// dq of one query tile (dq may be null) and, with part given, the tile's
// coefficient sums part[bh][it][kCo] = sum of ds {1, s_g, s_g s_h (g >= h)}.
__global__ __launch_bounds__(64 * kWvDq) void k64g_dq(const double* __restrict__ q, const double* __restrict__ k,
                                                    const double* __restrict__ v, const int32_t* __restrict__ labels,
                                                    const double* __restrict__ lam, const double* __restrict__ gam,
                                                    int G, int Hq, int Hkv, int N, double scale,
                                                    const double* __restrict__ Gv, const double* __restrict__ Gz,
                                                    double* __restrict__ dq, double* __restrict__ part) {
  __shared__ HeadTab tab;
  __shared__ double red[red_size(kWvDq)];
  __shared__ double cred[kWvDq][kCo];
  const int NT = (N + kM - 1) / kM, it = NT - 1 - (int)tile_of(blockIdx.y, blockIdx.z, gridDim.y);
  if (it < 0) return;
  const int bh = blockIdx.x, wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int b = bh / Hq, h = bh % Hq, u = b * Hkv + h / (Hq / Hkv);
  stage_head(tab, labels, nullptr, lam, gam, G, h);
  const int tq = it * kM + (lane & 15);
  const double* ku = k + (size_t)u * N * kD;
  const double* vu = v + (size_t)u * N * kD;
  double qr[16], gr[16];
  load_sorted(qr, q + (size_t)bh * N * kD, it * kM, N, tab, lane);
  load_rows(gr, Gv + (size_t)bh * N * kD, it * kM, N, lane);
  const double gz = Gz[(size_t)bh * N + (tq < N ? tq : N - 1)];
  d4 acc[4] = {};
  double co[kCo];
#pragma unroll
  for (int c = 0; c < kCo; ++c) co[c] = 0.0;
  for (int jt = wave; jt <= it; jt += kWvDq) {
    double kr[16], vr[16];
    load_sorted(kr, ku, jt * kM, N, tab, lane);
    load_rows(vr, vu, jt * kM, N, lane);
    d4 s[kG64], ds = {gz, gz, gz, gz};
    group_sums(s, kr, qr, scale, tab, lane);
#pragma unroll
    for (int x = 0; x < 16; ++x) ds = mma64(vr[x], gr[x], ds);
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int tk = jt * kM + 4 * r + (lane >> 4);
      ds[r] = tk <= tq && tk < N && tq < N ? ds[r] : 0.0;
    }
    if (dq) gradient_products(acc, s, ds * scale, ku, jt * kM, N, tab, lane);
    if (part) {
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        co[0] += ds[r];
#pragma unroll
        for (int g = 0; g < kG64; ++g) {
          const double x = ds[r] * s[g][r];
          co[1 + g] += x;
#pragma unroll
          for (int e = 0; e <= g; ++e)
            co[1 + kG64 + g * (g + 1) / 2 + e] = fma(x, s[e][r], co[1 + kG64 + g * (g + 1) / 2 + e]);
        }
      }
    }
  }
  if (part) {
#pragma unroll
    for (int c = 0; c < kCo; ++c) {
      double x = co[c];
#pragma unroll
      for (int off = 1; off < 64; off <<= 1) x += __shfl_xor(x, off, 64);
      if (lane == 0) cred[wave][c] = x;
    }
  }
  add_waves<kWvDq>(acc, red, wave, lane);
  if (part && threadIdx.x < kCo) {
    double x = 0.0;
    for (int w = 0; w < kWvDq; ++w) x += cred[w][threadIdx.x];
    part[((size_t)bh * NT + it) * kCo + threadIdx.x] = x;
  }
  if (wave || !dq) return;
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int row = it * kM + 4 * r + (lane >> 4);
    if (row >= N) continue;
#pragma unroll
    for (int cb = 0; cb < 4; ++cb) dq[((size_t)bh * N + row) * kD + tab.perm[16 * cb + (lane & 15)]] = acc[cb][r];
  }
}

// dk and dv of one key tile for one query head, into [B][Hq][N][64] (the heads
// of a unit are summed by k64g_headsum). Either may be null.
__global__ __launch_bounds__(64 * kWv) void k64g_dkv(const double* __restrict__ q, const double* __restrict__ k,
                                                     const double* __restrict__ v,
                                                     const int32_t* __restrict__ labels,
                                                     const double* __restrict__ c0, const double* __restrict__ lam,
                                                     const double* __restrict__ gam, int G, int Hq, int Hkv, int N,
                                                     double scale, const double* __restrict__ Gv,
                                                     const double* __restrict__ Gz, double* __restrict__ dkh,
                                                     double* __restrict__ dvh) {
  __shared__ HeadTab tab;
  __shared__ double red[red_size(kWv)];
  const int NT = (N + kM - 1) / kM, jt = (int)tile_of(blockIdx.y, blockIdx.z, gridDim.y);
  if (jt >= NT) return;
  const int bh = blockIdx.x, wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int b = bh / Hq, h = bh % Hq, u = b * Hkv + h / (Hq / Hkv);
  stage_head(tab, labels, c0, lam, gam, G, h);
  const int tk = jt * kM + (lane & 15);
  const double* qh = q + (size_t)bh * N * kD;
  const double* gh = Gv + (size_t)bh * N * kD;
  double kr[16], vr[16];
  load_sorted(kr, k + (size_t)u * N * kD, jt * kM, N, tab, lane);
  load_rows(vr, v + (size_t)u * N * kD, jt * kM, N, lane);
  d4 ak[4] = {}, av[4] = {};
  for (int it = jt + wave; it < NT; it += kWv) {
    double qr[16], gr[16];
    load_sorted(qr, qh, it * kM, N, tab, lane);
    load_rows(gr, gh, it * kM, N, lane);
    d4 s[kG64], ds;
    group_sums(s, qr, kr, scale, tab, lane);
    d4 kap = kappa_tile(s, tab);
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int tq = it * kM + 4 * r + (lane >> 4);
      ds[r] = Gz[(size_t)bh * N + (tq < N ? tq : N - 1)];
    }
#pragma unroll
    for (int x = 0; x < 16; ++x) ds = mma64(gr[x], vr[x], ds);
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int tq = it * kM + 4 * r + (lane >> 4);
      const bool ok = tk <= tq && tq < N && tk < N;
      kap[r] = ok ? kap[r] : 0.0;
      ds[r] = ok ? ds[r] * scale : 0.0;
    }
    if (dvh) value_products(av, kap, gh, it * kM, N, lane);
    if (dkh) gradient_products(ak, s, ds, qh, it * kM, N, tab, lane);
  }
  add_waves<kWv>(ak, red, wave, lane);
  add_waves<kWv>(av, red, wave, lane);
  if (wave) return;
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int row = jt * kM + 4 * r + (lane >> 4);
    if (row >= N) continue;
    const size_t o = ((size_t)bh * N + row) * kD;
#pragma unroll
    for (int cb = 0; cb < 4; ++cb) {
      const int c = 16 * cb + (lane & 15);
      if (dkh) dkh[o + tab.perm[c]] = ak[cb][r];
      if (dvh) dvh[o + c] = av[cb][r];
    }
  }
}

// dst[b][kv head][n][d] = sum over the unit's R query heads, in head order, of
// src[b][head][n][d]; blockIdx.y 0: (src0, dst0), 1: (src1, dst1).
__global__ __launch_bounds__(256) void k64g_headsum(const double* __restrict__ src0, const double* __restrict__ src1,
                                                    int R, size_t per_head, size_t total, double* __restrict__ dst0,
                                                    double* __restrict__ dst1) {
  const double* src = blockIdx.y ? src1 : src0;
  double* dst = blockIdx.y ? dst1 : dst0;
  const size_t x = (size_t)blockIdx.x * 256 + threadIdx.x;
  if (!dst || x >= total) return;
  const double* p = src + (x / per_head) * R * per_head + x % per_head;
  double acc = 0.0;
  for (int r = 0; r < R; ++r) acc += p[(size_t)r * per_head];
  dst[x] = acc;
}

// dc0, dlam, dgam of head h from the tiles' sums, added over (batch, tile): each
// wave a fixed share of them, lane by lane, then lanes and waves in a fixed order.
__global__ __launch_bounds__(256) void k64g_coef_grad(const double* __restrict__ part, int B, int Hq, int NT, int G,
                                                      double* __restrict__ dc0, double* __restrict__ dlam,
                                                      double* __restrict__ dgam) {
  __shared__ double w[kCo];
  const int h = blockIdx.x, wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  for (int c = wave; c < kCo; c += 4) {
    double x = 0.0;
    for (int i = lane; i < B * NT; i += 64) {
      const int b = i / NT, it = i % NT;
      x += part[((size_t)(b * Hq + h) * NT + it) * kCo + c];
    }
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) x += __shfl_xor(x, off, 64);
    if (lane == 0) w[c] = x;
  }
  __syncthreads();
  if (threadIdx.x == 0) dc0[h] = w[0];
  for (int e = threadIdx.x; e < G; e += 256) dlam[(size_t)h * G + e] = w[1 + e];
  for (int e = threadIdx.x; e < G * G; e += 256) {
    const int a = e / G, c = e % G, hi = a > c ? a : c, lo = a > c ? c : a;
    dgam[(size_t)h * G * G + e] = w[1 + kG64 + hi * (hi + 1) / 2 + lo];
  }
}

// ---------------------------------------------------------------------------
// Host launches.
// ---------------------------------------------------------------------------
size_t f64_workspace_bytes(const F64Geom& g, int G) {
  const int B = g.B, Hq = g.Hq, N = g.N;
  const size_t rows = (size_t)B * Hq * N;
  auto al = [](size_t x) { return (x + 255) & ~size_t(255); };
  const size_t grads = al(sizeof(double) * rows * kD) + al(sizeof(double) * rows);
  // group sums: dk and dv per query head where a unit has several, coefficient sums per 16-token tile
  if (G <= kG64)
    return grads + (Hq == g.Hkv ? 0 : 2 * al(sizeof(double) * rows * kD)) +
           al(sizeof(double) * B * Hq * ((N + kM - 1) / kM) * kCo);
  const size_t NT = (size_t)(N + kT - 1) / kT;
  return grads + al(sizeof(double) * B * Hq * NT * kFP);
}

void launch_f64_forward(const F64Geom& g, const double* q, const double* k, const double* v, const int32_t* labels,
                        const double* c0, const double* lam, const double* gam, int G, double scale, double* out,
                        double* num, double* den, hipStream_t st, const Timer& timed) {
  if (G <= kG64) {
    timed("k64g_fwd", st, [&] {
      const TileGrid t = tile_grid(g.B * g.Hq, (g.N + kM - 1) / kM);
      hipLaunchKernelGGL(k64g_fwd, dim3(t.x, t.y, t.z), dim3(64 * kWv), 0, st, q, k, v, labels, c0, lam, gam, G, g.Hq,
                         g.Hkv, g.N, scale, out, num, den);
    });
    return;
  }
  const int NT = (g.N + kT - 1) / kT;
  timed("k64_fwd", st, [&] {
    hipLaunchKernelGGL(k64_fwd, dim3(NT, g.B * g.Hq), dim3(kNT), 0, st, q, k, v, labels, c0, lam, gam, G, g.Hq,
                       g.Hkv, g.N, scale, out, num, den);
  });
}

void launch_f64_backward(const F64Geom& g, const double* q, const double* k, const double* v,
                         const int32_t* labels, const double* c0, const double* lam, const double* gam, int G,
                         double scale, const double* num, const double* den, const double* dout,
                         const double* dnum, const double* dden, double* dq, double* dk, double* dv, double* dc0,
                         double* dlam, double* dgam, void* workspace, hipStream_t st, const Timer& timed) {
  const size_t rows = (size_t)g.B * g.Hq * g.N;
  char* p = static_cast<char*>(workspace);
  auto take = [&](size_t n) {
    double* x = reinterpret_cast<double*>(p);
    p += (n * sizeof(double) + 255) & ~size_t(255);
    return x;
  };
  double* Gv = take(rows * kD);
  double* Gz = take(rows);
  timed("k64_gvec", st, [&] {
    hipLaunchKernelGGL(k64_gvec, dim3((unsigned)((rows + 3) / 4)), dim3(256), 0, st, dout, dnum, dden, num, den,
                       (long)rows, Gv, Gz);
  });
  if (G <= kG64) {
    const int NM = (g.N + kM - 1) / kM, R = g.Hq / g.Hkv;
    double* dkh = R > 1 ? take(rows * kD) : nullptr;
    double* dvh = R > 1 ? take(rows * kD) : nullptr;
    double* part = take((size_t)g.B * g.Hq * NM * kCo);
    const TileGrid t = tile_grid(g.B * g.Hq, NM);
    const dim3 grid(t.x, t.y, t.z);
    if (dq || dc0) {
      timed("k64g_dq", st, [&] {
        hipLaunchKernelGGL(k64g_dq, grid, dim3(64 * kWvDq), 0, st, q, k, v, labels, lam, gam, G, g.Hq, g.Hkv, g.N, scale, Gv, Gz,
                           dq, dc0 ? part : nullptr);
      });
    }
    if (dk || dv) {
      // one query head per KV head: the head's sums are the results
      double* dk1 = R == 1 ? dk : dk ? dkh : nullptr;
      double* dv1 = R == 1 ? dv : dv ? dvh : nullptr;
      timed("k64g_dkv", st, [&] {
        hipLaunchKernelGGL(k64g_dkv, grid, dim3(64 * kWv), 0, st, q, k, v, labels, c0, lam, gam, G, g.Hq, g.Hkv, g.N, scale,
                           Gv, Gz, dk1, dv1);
      });
      if (R > 1) {
        const size_t per_head = (size_t)g.N * kD, total = (size_t)g.B * g.Hkv * per_head;
        timed("k64g_headsum", st, [&] {
          hipLaunchKernelGGL(k64g_headsum, dim3((unsigned)((total + 255) / 256), 2), dim3(256), 0, st, dkh, dvh, R,
                             per_head, total, dk, dv);
        });
      }
    }
    if (dc0) {
      timed("k64g_coef_grad", st, [&] {
        hipLaunchKernelGGL(k64g_coef_grad, dim3(g.Hq), dim3(256), 0, st, part, g.B, g.Hq, NM, G, dc0, dlam, dgam);
      });
    }
    return;
  }
  const int NT = (g.N + kT - 1) / kT;
  double* part = take((size_t)g.B * g.Hq * NT * kFP);
  if (dq) {
    timed("k64_dq", st, [&] {
      hipLaunchKernelGGL(k64_dq, dim3(NT, g.B * g.Hq), dim3(kNT), 0, st, q, k, v, labels, lam, gam, G, g.Hq, g.Hkv,
                         g.N, scale, Gv, Gz, dq);
    });
  }
  if (dk || dv) {
    timed("k64_dkv", st, [&] {
      hipLaunchKernelGGL(k64_dkv, dim3(NT, g.B * g.Hkv), dim3(kNT), 0, st, q, k, v, labels, c0, lam, gam, G, g.Hq,
                         g.Hkv, g.N, scale, Gv, Gz, dk, dv);
    });
  }
  if (dc0) {
    timed("k64_coef_part", st, [&] {
      hipLaunchKernelGGL(k64_coef_part, dim3(NT, g.B * g.Hq), dim3(kCoefThreads), 0, st, q, k, v, g.Hq, g.Hkv, g.N,
                         scale, Gv, Gz, part);
    });
    timed("k64_coef_grad", st, [&] {
      hipLaunchKernelGGL(k64_coef_grad, dim3(g.Hq), dim3(256), 0, st, part, g.B, g.Hq, NT, labels, G, dc0, dlam,
                         dgam);
    });
  }
}

}  // namespace oal
