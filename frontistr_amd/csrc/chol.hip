// Factorization of the two-level step's coarse matrix E (FP64, SPD, banded) and the
// inverses its solves read, on the matrix cores.
//
// E is column-major with lda a multiple of 64 (unit diagonal in the padding) and is
// worked on in blocks of 64: block (i, j) is zero for i - j > w.
//  * Cholesky, right-looking: per block column one launch scales the panel by the
//    inverse of the diagonal block's factor, one updates the trailing band, and the
//    workgroup that updates the next diagonal block factors it in the same launch.
//    The band (11 blocks of 64 with six modes, 21 with twelve) is far too small to
//    fill the GPU: what bounds it is the chain of 5 + 35 us per block column, most of
//    it the 64 eliminations of the diagonal block.
//  * L^-1 and E^-1: column blocks of 16 are independent, so one workgroup per column
//    block substitutes forward down the band (T = L^-1) and, for E^-1, backward up
//    again (X = L^-T T, only the rows on and below the diagonal), with no
//    synchronization between workgroups.
// 1000 aggregates: 3.8 + 3.3 ms with six modes (order 6000, E^-1), 7.5 + 7.7 ms with
// twelve (order 12,000, L^-1); library calls per panel of 256 columns, then the dense
// inverse, took about 28 and 75 ms.
//
// v_mfma_f64_16x16x4: lane l holds A[l % 16][l / 16], B[l / 16][l % 16] and, as its
// i-th result, D[4 i + l / 16][l % 16].  Which operand takes which factor is chosen
// so that sixteen lanes load or store sixteen consecutive doubles.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>

#include "device.h"

namespace hecmw33 {
namespace {

typedef double v4d __attribute__((ext_vector_type(4)));
constexpr int kNB = 64;
constexpr int kCholBlock = 256;

__device__ __forceinline__ v4d mfma(double a, double b, v4d c) {
  return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}

// 1 / d to the last bit or two: the hardware estimate and two Newton steps
__device__ __forceinline__ double recip(double d) {
  double r = __builtin_amdgcn_rcp(d);
  r = fma(r, fma(-d, r, 1.0), r);
  return fma(r, fma(-d, r, 1.0), r);
}

// acc -= P Q^T for this wave's 32 x 32 quadrant (rows c of P against rows r of Q,
// D[c][r]), P and Q column-major 64 x 64 at p, q
__device__ __forceinline__ void quad_product(const double* __restrict__ p, const double* __restrict__ q, int64_t ldp,
                                             int64_t ldq, int l, v4d (&acc)[2][2]) {
  double a[2][16], b[2][16];
#pragma unroll
  for (int s = 0; s < 16; ++s) {
    const int m = 4 * s + l / 16;
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      a[t][s] = p[16 * t + l % 16 + m * ldp];
      b[t][s] = q[16 * t + l % 16 + m * ldq];
    }
  }
#pragma unroll
  for (int s = 0; s < 16; ++s)
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int u = 0; u < 2; ++u) acc[t][u] = mfma(a[t][s], b[u][s], acc[t][u]);
}

// Linv (column-major) = inverse of the Cholesky factor of the 64 x 64 block M:
// eliminations on a 4 x 4 tile per thread, with the pivot row and column passed
// through LDS.  Column j turns from the Schur complement into column j of the
// inverse of the unit factor at step j, so one array holds both.
__device__ __forceinline__ void factor_block(double (&m)[4][4], double* __restrict__ Linv, int32_t* info) {
  __shared__ double prow[2][kNB], pcol[2][kNB], diag[kNB];
  const int ti = threadIdx.x / 16, tj = threadIdx.x % 16;
  bool bad = false;
  for (int j4 = 0; j4 < 16; ++j4)
#pragma unroll
    for (int jj = 0; jj < 4; ++jj) {
      const int j = 4 * j4 + jj, buf = jj & 1;
      if (ti == j4)
#pragma unroll
        for (int c = 0; c < 4; ++c) prow[buf][4 * tj + c] = m[jj][c];
      if (tj == j4)
#pragma unroll
        for (int r = 0; r < 4; ++r) pcol[buf][4 * ti + r] = m[r][jj];
      __syncthreads();
      double d = prow[buf][j];
      if (!(d > 0.0) || !(d < 1e308)) {
        bad = true;
        d = 1.0;
      }
      if (threadIdx.x == 0) diag[j] = d;
      const double rd = recip(d);
      double row[4];
#pragma unroll
      for (int c = 0; c < 4; ++c) row[c] = 4 * tj + c == j ? 1.0 : prow[buf][4 * tj + c];
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        if (4 * ti + r <= j) continue;
        const double f = pcol[buf][4 * ti + r] * rd;
#pragma unroll
        for (int c = 0; c < 4; ++c) m[r][c] = (4 * tj + c == j ? 0.0 : m[r][c]) - f * row[c];
      }
      if (ti == j4 && tj == j4) m[jj][jj] = 1.0;
    }
  __syncthreads();
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const double s = 1.0 / sqrt(diag[4 * ti + r]);
#pragma unroll
    for (int c = 0; c < 4; ++c)
      Linv[4 * ti + r + kNB * (4 * tj + c)] = 4 * ti + r >= 4 * tj + c ? s * m[r][c] : 0.0;
  }
  if (bad && threadIdx.x == 0) *info = 1;
}

__global__ __launch_bounds__(kCholBlock) void k_chol_first(const double* __restrict__ E, int64_t lda,
                                                            double* __restrict__ Linv, int32_t* info) {
  double m[4][4];
  const int ti = threadIdx.x / 16, tj = threadIdx.x % 16;
#pragma unroll
  for (int r = 0; r < 4; ++r)
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      const int i = 4 * ti + r, k = 4 * tj + c;
      m[r][c] = E[max(i, k) + min(i, k) * lda];
    }
  factor_block(m, Linv, info);
}

// L_ik = A_ik Linv_k^T for the blocks i = k + 1 + blockIdx.x of panel k, in place
__global__ __launch_bounds__(kCholBlock) void k_chol_panel(double* __restrict__ E, int64_t lda, int k,
                                                            const double* __restrict__ Linv) {
  const int l = threadIdx.x % 64, w = threadIdx.x / 64, c0 = 32 * (w / 2), r0 = 32 * (w % 2);
  double* blk = E + (int64_t)kNB * (k + 1 + blockIdx.x) + (int64_t)kNB * k * lda;
  v4d acc[2][2] = {};
  quad_product(Linv + (int64_t)kNB * kNB * k + c0, blk + r0, kNB, lda, l, acc);
  __syncthreads();  // every wave has read its rows
#pragma unroll
  for (int t = 0; t < 2; ++t)
#pragma unroll
    for (int u = 0; u < 2; ++u)
#pragma unroll
      for (int i = 0; i < 4; ++i)
        blk[r0 + 16 * u + l % 16 + (int64_t)(c0 + 16 * t + 4 * i + l / 16) * lda] = acc[t][u][i];
}

// A_ij -= L_ik L_jk^T for the blocks k < j <= i of panel k's band (blockIdx.x: the
// pairs by rows); the first, (k+1, k+1), is then factored
__global__ __launch_bounds__(kCholBlock) void k_chol_update(double* __restrict__ E, int64_t lda, int k,
                                                             double* __restrict__ Linv, int32_t* info) {
  const int l = threadIdx.x % 64, w = threadIdx.x / 64, c0 = 32 * (w / 2), r0 = 32 * (w % 2);
  int i = 0, rest = blockIdx.x;
  while (rest > i) {
    rest -= i + 1;
    ++i;
  }
  const int bi = k + 1 + i, bj = k + 1 + rest;
  const double* pan = E + (int64_t)kNB * k * lda;
  double* blk = E + (int64_t)kNB * bi + (int64_t)kNB * bj * lda;
  v4d acc[2][2] = {};
  quad_product(pan + (int64_t)kNB * bj + c0, pan + (int64_t)kNB * bi + r0, lda, lda, l, acc);
  __shared__ double tile[kNB * (kNB + 1)];
  const bool next = blockIdx.x == 0;
#pragma unroll
  for (int t = 0; t < 2; ++t)
#pragma unroll
    for (int u = 0; u < 2; ++u)
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int r = r0 + 16 * u + l % 16, c = c0 + 16 * t + 4 * q + l / 16;
        const int64_t at = r + (int64_t)c * lda;
        const double v = blk[at] - acc[t][u][q];
        if (next)
          tile[r + c * (kNB + 1)] = v;
        else
          blk[at] = v;
      }
  if (!next) return;
  __syncthreads();
  double m[4][4];
  const int ti = threadIdx.x / 16, tj = threadIdx.x % 16;
#pragma unroll
  for (int r = 0; r < 4; ++r)
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      const int y = 4 * ti + r, x = 4 * tj + c;
      m[r][c] = tile[max(y, x) + min(y, x) * (kNB + 1)];
    }
  factor_block(m, Linv + (int64_t)kNB * kNB * (k + 1), info);
}

// One 64 x 64 block against the 64 x 16 block row y (row-major at y, stride ldy):
// acc -= P y for this wave's 16 rows.  TRANS: P = B^T with B column-major at b, its
// sixteen-row runs loaded as they lie (lane l takes rows 16 s + 4 (l/16) + t of
// column l % 16 in MFMA step t, and the same rows of y).
template <bool TRANS>
struct Frags {
  double a[16], b[16];
  __device__ __forceinline__ void load(const double* __restrict__ p, int64_t ldp, const double* __restrict__ y,
                                       int64_t ldy, int l, int wave) {
#pragma unroll
    for (int s = 0; s < 16; ++s) {
      if (TRANS) {
        const int m = 16 * (s / 4) + 4 * (l / 16) + s % 4;
        a[s] = p[m + (int64_t)(16 * wave + l % 16) * ldp];
        b[s] = y[(int64_t)m * ldy + l % 16];
      } else {
        const int m = 4 * s + l / 16;
        a[s] = p[16 * wave + l % 16 + (int64_t)m * ldp];
        b[s] = y[(int64_t)m * ldy + l % 16];
      }
    }
  }
  __device__ __forceinline__ void apply(v4d& acc) const {
#pragma unroll
    for (int s = 0; s < 16; ++s) acc = mfma(a[s], b[s], acc);
  }
};

// One step of a substitution: block row i of the 16 columns at c0, y = base (its
// old content or the identity) - sum over j of P_ij (row j), then the product with
// the diagonal block's inverse factor.  Rows live in E's upper triangle, row-major:
// (r, c) at E[c + r lda].
template <bool TRANS>
__device__ __forceinline__ void substitute(double* __restrict__ E, int64_t lda, const double* __restrict__ Linv, int i,
                                           int j0, int j1, int c0, bool identity, double* __restrict__ ly) {
  const int l = threadIdx.x % 64, wave = threadIdx.x / 64;
  v4d acc = {0.0, 0.0, 0.0, 0.0};
  auto block = [&](int j) { return TRANS ? E + (int64_t)kNB * j + (int64_t)kNB * i * lda : E + (int64_t)kNB * i + (int64_t)kNB * j * lda; };
  auto rows = [&](int j) { return E + c0 + (int64_t)kNB * j * lda; };
  // the next block's loads in flight during the present one's products
  Frags<TRANS> f, g;
  if (j0 < j1) f.load(block(j0), lda, rows(j0), lda, l, wave);
  for (int j = j0; j < j1; j += 2) {
    if (j + 1 < j1) g.load(block(j + 1), lda, rows(j + 1), lda, l, wave);
    f.apply(acc);
    if (j + 1 < j1) {
      if (j + 2 < j1) f.load(block(j + 2), lda, rows(j + 2), lda, l, wave);
      g.apply(acc);
    }
  }
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const int r = 16 * wave + 4 * q + l / 16, c = l % 16;
    const double base = identity ? (kNB * i + r == c0 + c ? 1.0 : 0.0) : (TRANS ? rows(i)[c + (int64_t)r * lda] : 0.0);
    ly[r * 16 + c] = base - acc[q];
  }
  __syncthreads();
  v4d out = {0.0, 0.0, 0.0, 0.0};
  Frags<TRANS> d;
  d.load(Linv + (int64_t)kNB * kNB * i, kNB, ly, 16, l, wave);
  d.apply(out);
#pragma unroll
  for (int q = 0; q < 4; ++q) rows(i)[l % 16 + (int64_t)(16 * wave + 4 * q + l / 16) * lda] = out[q];
  __syncthreads();  // the rows are in memory for the next step, ly is free
}

// columns 16 blockIdx.x .. + 15 of T = L^-1, and with `both` of X = L^-T T
__global__ __launch_bounds__(kCholBlock) void k_chol_inverse(double* __restrict__ E, int64_t lda,
                                                              const double* __restrict__ Linv, int nb, int w,
                                                              int both) {
  __shared__ double ly[kNB * 16];
  const int c0 = 16 * blockIdx.x, kc = c0 / kNB;
  for (int i = kc; i < nb; ++i) substitute<false>(E, lda, Linv, i, max(kc, i - w), i, c0, i == kc, ly);
  if (!both) return;
  for (int i = nb - 1; i >= kc; --i) substitute<true>(E, lda, Linv, i, i + 1, min(nb, i + w + 1), c0, false, ly);
}

__global__ void k_chol_pad(double* __restrict__ E, int64_t lda, int n, int np) {
  const int i = n + blockIdx.x * blockDim.x + threadIdx.x;
  if (i < np) E[i + i * lda] = 1.0;
}

}  // namespace

int32_t coarse_padded(int32_t nc) { return (nc + kNB - 1) / kNB * kNB; }

// E (column-major, order nc padded to np = lda, half bandwidth `band`) -> in its upper
// triangle, row-major, L^-1 (both = false) or E^-1.  Linv: np * 64 doubles; *info is
// set when E is not positive definite (clear before).
void coarse_factor(double* E, int32_t nc, int32_t band, double* Linv, bool both, int32_t* info, hipStream_t s) {
  const int32_t np = coarse_padded(nc), nb = np / kNB, w = std::min((band + kNB - 1) / kNB, nb - 1);
  if (np > nc) k_chol_pad<<<1, kNB, 0, s>>>(E, np, nc, np);
  k_chol_first<<<1, kCholBlock, 0, s>>>(E, np, Linv, info);
  for (int32_t k = 0; k + 1 < nb; ++k) {
    const int32_t m = std::max(1, std::min(w, nb - 1 - k));
    k_chol_panel<<<m, kCholBlock, 0, s>>>(E, np, k, Linv);
    k_chol_update<<<m * (m + 1) / 2, kCholBlock, 0, s>>>(E, np, k, Linv, info);
  }
  k_chol_inverse<<<np / 16, kCholBlock, 0, s>>>(E, np, Linv, nb, w, both ? 1 : 0);
}

}  // namespace hecmw33
