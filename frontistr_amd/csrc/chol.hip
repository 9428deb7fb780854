// Factorization of the two-level step's coarse matrix E (FP64, SPD, banded) and the
// inverses its solves read, on the matrix cores.
//
// E is worked on in blocks of 64, of which those of the band's w + 1 block diagonals are
// stored, each by itself, so that a block's loads are consecutive (with the dense
// matrix's column stride they touched a page per column).
//  * Cholesky, right-looking: per block column one launch scales the panel by the
//    inverse of the diagonal block's factor, one updates the trailing band, and the
//    workgroup that updates the next diagonal block factors it in the same launch.
//    The band (11 blocks of 64 with six modes, 21 with twelve) is far too small to
//    fill the GPU: what bounds it is the chain of 5 + 28 us per block column, 20 of
//    them the 64 eliminations of the diagonal block.
//  * L^-1 and E^-1: column blocks of 16 are independent, so one workgroup per column
//    block substitutes forward down the band (T = L^-1) and, for E^-1, backward up
//    again (X = L^-T T, only the rows on and below the diagonal), with no
//    synchronization between workgroups.  The chain of the longest column bounds it,
//    14 us per block row.
// 1000 aggregates: 3.1 + 2.7 ms with six modes (order 6000, E^-1), 6.3 + 6.7 ms with
// twelve (order 12,000, L^-1); with the band in a dense column-major array, four waves
// per column block and a barrier per eliminated column 3.8 + 3.3 and 7.5 + 7.7; library
// calls per panel of 256 columns, then the dense inverse, took about 28 and 75 ms.
//
// v_mfma_f64_16x16x4: lane l holds A[l % 16][l / 16], B[l / 16][l % 16] and, as its
// i-th result, D[4 i + l / 16][l % 16].  Which operand takes which factor is chosen
// so that sixteen lanes load or store sixteen consecutive doubles.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>

#include "device.h"
#include "resident.h"

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
__device__ __forceinline__ void quad_product(const double* __restrict__ p, const double* __restrict__ q, int l,
                                             v4d (&acc)[2][2]) {
  double a[2][16], b[2][16];
#pragma unroll
  for (int s = 0; s < 16; ++s) {
    const int m = 4 * s + l / 16;
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      a[t][s] = p[16 * t + l % 16 + m * kNB];
      b[t][s] = q[16 * t + l % 16 + m * kNB];
    }
  }
#pragma unroll
  for (int s = 0; s < 16; ++s)
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int u = 0; u < 2; ++u) acc[t][u] = mfma(a[t][s], b[u][s], acc[t][u]);
}

__device__ __forceinline__ double readlane(double v, int lane) {
  return __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(v), lane),
                          __builtin_amdgcn_readlane(__double2loint(v), lane));
}

// Linv (column-major) = inverse of the Cholesky factor of the 64 x 64 block in LDS, M(r, c)
// at tile[r + kTile c], r >= c, and both triangles of the 16 x 16 diagonal blocks.
// L D L^T by panels of 16 columns: a wave eliminates a panel with a row per lane, the
// pivot rows by readlane and no barrier; rank-16 products on the matrix cores update
// what remains.  The inverse of the unit factor, X, goes transposed into the upper
// triangle: the diagonal blocks by substitution beside the next panel, then block
// diagonal by block diagonal X_ij = -X_ii sum L_ik X_kj.  20 us, 13 of them the four
// panels (0.2 us per column: the pivot's reciprocal and the row's readlanes); with a
// barrier per column on a tile per thread 27.
constexpr int kTile = kNB + 1, kPanel = 16, kG = kPanel + 1;
__device__ __forceinline__ void factor_block(double* __restrict__ tile, double* __restrict__ g, double* __restrict__ diag,
                                             double* __restrict__ Linv, int32_t* info) {
  const int l = threadIdx.x % 64, w = __builtin_amdgcn_readfirstlane(threadIdx.x / 64), lr = l % 16, lk = l / 16;
  constexpr int kP = kNB / kPanel;
  auto at = [&](int r, int c) -> double& { return tile[r + kTile * c]; };
  // X of diagonal block b, a column per lane, and the scales of its rows
  auto invert_diagonal = [&](int b) {
    if (l >= kPanel) return;
    const int o = kPanel * b;
    diag[o + l] = 1.0 / sqrt(diag[o + l]);
    double x[kPanel];
#pragma unroll
    for (int r = 0; r < kPanel; ++r) x[r] = r == l ? 1.0 : 0.0;
#pragma unroll
    for (int k = 0; k < kPanel - 1; ++k)
#pragma unroll
      for (int r = k + 1; r < kPanel; ++r) x[r] = fma(-at(o + r, o + k), x[k], x[r]);
    lds_order();
#pragma unroll
    for (int r = 0; r < kPanel; ++r)
      if (r >= l) at(o + l, o + r) = x[r];
  };
#pragma unroll 1
  for (int p = 0; p <= kP; ++p) {
    const int c0 = kPanel * p;
    if (w == p) {
      // one stretch of code without a branch, so that a pivot's reciprocal is under way
      // while the columns behind it are updated
      double m[kPanel], f[kPanel], own = 1.0;
      bool bad = false;
#pragma unroll
      for (int c = 0; c < kPanel; ++c) m[c] = at(l, c0 + c);
#pragma unroll
      for (int j = 0; j < kPanel; ++j) {
        double d = readlane(m[j], c0 + j);
        const bool no = !(d > 0.0) || !(d < 1e308);
        bad |= no;
        d = no ? 1.0 : d;
        own = l == c0 + j ? d : own;
        f[j] = l > c0 + j ? m[j] * recip(d) : 0.0;
#pragma unroll
        for (int c = j + 1; c < kPanel; ++c) m[c] = fma(-f[j], readlane(m[c], c0 + j), m[c]);
      }
#pragma unroll
      for (int j = 0; j < kPanel; ++j) {
        g[l * kG + j] = m[j];
        if (l > c0 + j) at(l, c0 + j) = f[j];
      }
      if (l >= c0 && l < c0 + kPanel) diag[l] = own;
      if (bad && l == 0) *info = 1;
    } else if (w == p - 1) {
      invert_diagonal(p - 1);
    }
    __syncthreads();
    // A_ij -= F_i G_j^T, tiles p < j <= i dealt to the waves
    int t = 0;
    for (int i = p + 1; i < kP; ++i)
      for (int j = p + 1; j <= i; ++j, ++t) {
        if (t % kP != w) continue;
        v4d acc = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
        for (int s = 0; s < kPanel / 4; ++s)
          acc = mfma(at(kPanel * i + lr, c0 + 4 * s + lk), g[(kPanel * j + lr) * kG + 4 * s + lk], acc);
#pragma unroll
        for (int q = 0; q < 4; ++q) at(kPanel * i + 4 * q + lk, kPanel * j + lr) -= acc[q];
      }
    __syncthreads();
  }
#pragma unroll 1
  for (int d = 1; d < kP; ++d) {
    const int i = w + d, j = w;
    if (i < kP) {
      v4d sum = {0.0, 0.0, 0.0, 0.0}, x = {0.0, 0.0, 0.0, 0.0};
      for (int k = j; k < i; ++k)
#pragma unroll
        for (int s = 0; s < kPanel / 4; ++s) {
          const int kk = 4 * s + lk;
          const double b = k > j || kk >= lr ? at(kPanel * j + lr, kPanel * k + kk) : 0.0;
          sum = mfma(at(kPanel * i + lr, kPanel * k + kk), b, sum);
        }
#pragma unroll
      for (int s = 0; s < kPanel / 4; ++s) {
        const int kk = 4 * s + lk;
        x = mfma(lr >= kk ? at(kPanel * i + kk, kPanel * i + lr) : 0.0, sum[s], x);
      }
#pragma unroll
      for (int q = 0; q < 4; ++q) at(kPanel * j + lr, kPanel * i + 4 * q + lk) = -x[q];
    }
    __syncthreads();
  }
  const int r = threadIdx.x % kNB;
  for (int c = threadIdx.x / kNB; c < kNB; c += kCholBlock / kNB) Linv[r + kNB * c] = r >= c ? at(c, r) * diag[r] : 0.0;
}

__global__ __launch_bounds__(kCholBlock) void k_chol_first(const double* __restrict__ E, double* __restrict__ Linv,
                                                            int32_t* info) {
  __shared__ double tile[kNB * kTile], g[kNB * kG], diag[kNB];
  for (int k = threadIdx.x; k < kNB * kNB; k += kCholBlock) {
    const int r = k % kNB, c = k / kNB;
    tile[r + kTile * c] = E[max(r, c) + kNB * min(r, c)];
  }
  __syncthreads();
  factor_block(tile, g, diag, Linv, info);
}

// block (i, j) of the band
__device__ __forceinline__ double* block(double* E, int w, int i, int j) {
  return E + ((int64_t)j * (w + 1) + i - j) * (kNB * kNB);
}

// L_ik = A_ik Linv_k^T for the blocks i = k + 1 + blockIdx.x of panel k, in place
__global__ __launch_bounds__(kCholBlock) void k_chol_panel(double* __restrict__ E, int bw, int k,
                                                            const double* __restrict__ Linv) {
  const int l = threadIdx.x % 64, w = threadIdx.x / 64, c0 = 32 * (w / 2), r0 = 32 * (w % 2);
  double* blk = block(E, bw, k + 1 + blockIdx.x, k);
  v4d acc[2][2] = {};
  quad_product(Linv + (int64_t)kNB * kNB * k + c0, blk + r0, l, acc);
  __syncthreads();  // every wave has read its rows
#pragma unroll
  for (int t = 0; t < 2; ++t)
#pragma unroll
    for (int u = 0; u < 2; ++u)
#pragma unroll
      for (int i = 0; i < 4; ++i) blk[r0 + 16 * u + l % 16 + (c0 + 16 * t + 4 * i + l / 16) * kNB] = acc[t][u][i];
}

// A_ij -= L_ik L_jk^T for the blocks k < j <= i of panel k's band (blockIdx.x: the
// pairs by rows); the first, (k+1, k+1), is then factored
__global__ __launch_bounds__(kCholBlock) void k_chol_update(double* __restrict__ E, int bw, int k,
                                                             double* __restrict__ Linv, int32_t* info) {
  const int l = threadIdx.x % 64, w = threadIdx.x / 64, c0 = 32 * (w / 2), r0 = 32 * (w % 2);
  int i = 0, rest = blockIdx.x;
  while (rest > i) {
    rest -= i + 1;
    ++i;
  }
  const int bi = k + 1 + i, bj = k + 1 + rest;
  double* blk = block(E, bw, bi, bj);
  v4d acc[2][2] = {};
  quad_product(block(E, bw, bj, k) + c0, block(E, bw, bi, k) + r0, l, acc);
  __shared__ double tile[kNB * kTile], g[kNB * kG], diag[kNB];
  const bool next = blockIdx.x == 0;
#pragma unroll
  for (int t = 0; t < 2; ++t)
#pragma unroll
    for (int u = 0; u < 2; ++u)
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int r = r0 + 16 * u + l % 16, c = c0 + 16 * t + 4 * q + l / 16;
        const int at = r + c * kNB;
        if (!next) {
          blk[at] -= acc[t][u][q];
        } else if (r >= c) {
          const double v = blk[at] - acc[t][u][q];
          tile[r + kTile * c] = v;
          tile[c + kTile * r] = v;
        }
      }
  if (!next) return;
  __syncthreads();
  factor_block(tile, g, diag, Linv + (int64_t)kNB * kNB * (k + 1), info);
}

// k_chol_inverse: kInvCols columns by kInvSplit groups of four waves
constexpr int kInvCols = 16, kInvSplit = 4;

// One 64 x 64 block P against the 64 x kInvCols block row y (row-major): acc += P y for
// this wave's 16 rows.  TRANS: P = B^T with B column-major at p, its sixteen-row runs
// loaded as they lie (lane l takes rows 16 s + 4 (l/16) + t of column l % 16 in
// MFMA step t, and the same rows of y).
template <bool TRANS>
struct Frags {
  double a[16], b[16];
  static __device__ __forceinline__ int inner(int s, int l) { return TRANS ? 16 * (s / 4) + 4 * (l / 16) + s % 4 : 4 * s + l / 16; }
  __device__ __forceinline__ void load_p(const double* __restrict__ p, int l, int rows) {
#pragma unroll
    for (int s = 0; s < 16; ++s) {
      const int m = inner(s, l), r = 16 * rows + l % 16;
      a[s] = TRANS ? p[m + r * kNB] : p[r + m * kNB];
    }
  }
  __device__ __forceinline__ void load_y(const double* __restrict__ y, int l) {
#pragma unroll
    for (int s = 0; s < 16; ++s) b[s] = y[inner(s, l) * kInvCols + l % 16];
  }
  __device__ __forceinline__ void apply(v4d& acc) const {
#pragma unroll
    for (int s = 0; s < 16; ++s) acc = mfma(a[s], b[s], acc);
  }
};

// One step of a substitution: block row i of the columns whose rows are at T, y = base
// (its old content or the identity from column d0 of the block on) - sum over j of P_ij
// (row j), then the product with the diagonal block's inverse factor.  The blocks j
// are dealt to the groups of waves: what a step takes is the loads of the blocks that
// follow each other in a wave.
template <bool TRANS>
__device__ __forceinline__ void substitute(double* __restrict__ T, double* __restrict__ E, const double* __restrict__ Linv,
                                           int bw, int i, int j0, int j1, int d0, double (*part)[kNB * kInvCols]) {
  const int l = threadIdx.x % 64, wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64), rw = wave % 4, group = wave / 4;
  v4d acc = {0.0, 0.0, 0.0, 0.0};
  double* const row = T + (int64_t)kNB * kInvCols * i;
  Frags<TRANS> f;
#pragma unroll 1
  for (int j = j0 + group; j < j1; j += kInvSplit) {
    f.load_p(TRANS ? block(E, bw, j, i) : block(E, bw, i, j), l, rw);
    f.load_y(T + (int64_t)kNB * kInvCols * j, l);
    f.apply(acc);
  }
  if (group == 0) f.load_p(Linv + (int64_t)kNB * kNB * i, l, rw);
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const int r = 16 * rw + 4 * q + l / 16, c = l % 16;
    double base = 0.0;
    if (group == 0) base = TRANS ? row[r * kInvCols + c] : (r == d0 + c ? 1.0 : 0.0);
    part[group][r * kInvCols + c] = base - acc[q];
  }
  __syncthreads();
  if (group == 0) {
    f.load_y(part[0], l);
    for (int g = 1; g < kInvSplit; ++g)
#pragma unroll
      for (int s = 0; s < 16; ++s) f.b[s] += part[g][f.inner(s, l) * kInvCols + l % 16];
    v4d out = {0.0, 0.0, 0.0, 0.0};
    f.apply(out);
#pragma unroll
    for (int q = 0; q < 4; ++q) row[(16 * rw + 4 * q + l / 16) * kInvCols + l % 16] = out[q];
  }
  __syncthreads();  // the rows are in memory for the next step, part is free
}

// kInvCols columns of T = L^-1, and with `both` of X = L^-T T
__global__ __launch_bounds__(kInvSplit * kCholBlock) void k_chol_inverse(double* __restrict__ E, double* __restrict__ T,
                                                                          const double* __restrict__ Linv, int nb,
                                                                          int bw, int both) {
  __shared__ double part[kInvSplit][kNB * kInvCols];
  // the workgroups of a block column share an XCD and so its L2: the blocks of L that
  // they read at the same time come from memory once
  constexpr int kPer = kNB / kInvCols;
  const int xcd = blockIdx.x % kNumXcd, local = blockIdx.x / kNumXcd, kc = local / kPer * kNumXcd + xcd;
  if (kc >= nb) return;
  double* const t = T + (int64_t)(kPer * kc + local % kPer) * nb * (kNB * kInvCols);
  for (int i = kc; i < nb; ++i)
    substitute<false>(t, E, Linv, bw, i, max(kc, i - bw), i, i == kc ? kInvCols * (local % kPer) : kNB, part);
  if (!both) return;
  for (int i = nb - 1; i >= kc; --i) substitute<true>(t, E, Linv, bw, i, i + 1, min(nb, i + bw + 1), 0, part);
}

}  // namespace

// E (band blocks, unit diagonal in the padding) -> T: L^-1 (both = false) or E^-1; see device.h
void coarse_factor(const CoarseBand& e, double* Linv, double* T, bool both, int32_t* info, hipStream_t s) {
  const int32_t nb = e.np / kNB;
  k_chol_first<<<1, kCholBlock, 0, s>>>(e.E, Linv, info);
  for (int32_t k = 0; k + 1 < nb; ++k) {
    const int32_t m = std::min(e.w, nb - 1 - k);
    if (m < 1) {
      // a band inside the diagonal blocks
      k_chol_first<<<1, kCholBlock, 0, s>>>(e.E + (int64_t)kNB * kNB * (k + 1), Linv + (int64_t)kNB * kNB * (k + 1), info);
      continue;
    }
    k_chol_panel<<<m, kCholBlock, 0, s>>>(e.E, e.w, k, Linv);
    k_chol_update<<<m * (m + 1) / 2, kCholBlock, 0, s>>>(e.E, e.w, k, Linv, info);
  }
  k_chol_inverse<<<kNB / kInvCols * ((nb + kNumXcd - 1) / kNumXcd * kNumXcd), kInvSplit * kCholBlock, 0, s>>>(e.E, T, Linv, nb, e.w,
                                                                                                         both ? 1 : 0);
}

}  // namespace hecmw33
