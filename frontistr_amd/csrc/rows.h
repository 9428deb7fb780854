// Device code that several kernel files share: block numbering, wave sums, the
// SpMV row product and the 3x3 LU solve.
#pragma once
#include <hip/hip_runtime.h>

#include <cstdint>

#include "device.h"

namespace hecmw33 {

__device__ __forceinline__ int xcd_block(int bid, int nblk) {
  // Workgroups are dealt to the 8 XCDs round-robin; give each XCD a contiguous
  // run of logical blocks so neighbouring slices share that XCD's L2.
  const int xcd = bid % kNumXcd, local = bid / kNumXcd;
  const int per = nblk / kNumXcd, rem = nblk % kNumXcd;
  return xcd < rem ? xcd * (per + 1) + local : rem * (per + 1) + (xcd - rem) * per + local;
}

__device__ __forceinline__ double wave_sum(double v) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, kWave);
  return v;
}

__device__ __forceinline__ int lane_id() { return threadIdx.x & (kWave - 1); }

// aval_load past the caches' replacement
__device__ __forceinline__ void aval_load_nt(const double* __restrict__ val, int64_t g, int r, double (&v)[9]) {
  typedef double D2 __attribute__((ext_vector_type(2)));
  const double* __restrict__ b = val + g * (9 * kRowsA);
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const D2 t = __builtin_nontemporal_load(reinterpret_cast<const D2*>(b + q * (2 * kRowsA) + 2 * r));
    v[2 * q] = t.x;
    v[2 * q + 1] = t.y;
  }
  v[8] = __builtin_nontemporal_load(b + 8 * kRowsA + r);
}

constexpr int kSpmvChunk = 4;

// SpMV rows, SELL-64, one row per lane (kRowsA).  FP64 in the reference's
// order: the D block first, then L, then U in storage order;
// y = ((y + a1*x1) + a2*x2) + a3*x3, no fused multiply-add.  A chunk of U
// blocks is loaded before it is accumulated in order; the D block is slot 0
// of the first chunk, so no load waits for a block of its own.  y starts at
// -0, for which -0 + a is a exactly (also for a = -0), so the D block's sum is
// the reference's (a1*x1 + a2*x2) + a3*x3.  xo = x of the row itself.
// One chunk of U blocks from k0.  FULL: every block is live, so no load or sum
// of the chunk sits under a condition and all its loads are in flight
// together (a per-block condition lets the compiler move a block's loads into
// a branch of their own, one more dependent round trip per chunk).  Not FULL
// (the row's last chunk): slots past the end re-read the last block and are
// masked out of the sum.
template <int U, bool FULL, bool NT>
__device__ __forceinline__ void sell_chunk(const Sell<double>& a, int base, int lane, const int32_t* __restrict__ colp,
                                           const double* __restrict__ x, int k0, int len, double (&y)[3],
                                           double (&xo)[3]) {
#pragma clang fp contract(off)
  int kk[U], c[U];
#pragma unroll
  for (int j = 0; j < U; ++j) {
    kk[j] = (FULL || k0 + j < len) ? k0 + j : len - 1;
    c[j] = NT ? __builtin_nontemporal_load(colp + (int64_t)kk[j] * kRowsA) : colp[(int64_t)kk[j] * kRowsA];
  }
  double v[U][9], xv[U][3];
#pragma unroll
  for (int j = 0; j < U; ++j) {
    if (NT)
      aval_load_nt(a.val, (int64_t)base + kk[j], lane, v[j]);
    else
      aval_load(a.val, (int64_t)base + kk[j], lane, v[j]);
    xv[j][0] = x[3 * (int64_t)c[j]];
    xv[j][1] = x[3 * (int64_t)c[j] + 1];
    xv[j][2] = x[3 * (int64_t)c[j] + 2];
  }
  if (k0 == 0) {
    xo[0] = xv[0][0];
    xo[1] = xv[0][1];
    xo[2] = xv[0][2];
  }
#pragma unroll
  for (int j = 0; j < U; ++j) {
    const double t0 = y[0] + v[j][0] * xv[j][0] + v[j][1] * xv[j][1] + v[j][2] * xv[j][2];
    const double t1 = y[1] + v[j][3] * xv[j][0] + v[j][4] * xv[j][1] + v[j][5] * xv[j][2];
    const double t2 = y[2] + v[j][6] * xv[j][0] + v[j][7] * xv[j][1] + v[j][8] * xv[j][2];
    if (FULL) {
      y[0] = t0;
      y[1] = t1;
      y[2] = t2;
    } else {
      const bool live = k0 + j < len;
      y[0] = live ? t0 : y[0];
      y[1] = live ? t1 : y[1];
      y[2] = live ? t2 : y[2];
    }
  }
}

template <int U, bool NT = false>
__device__ __forceinline__ void sell_row(const Sell<double>& a, int s, int lane, const double* __restrict__ x,
                                         double (&y)[3], double (&xo)[3]) {
#pragma clang fp contract(off)
  const int base = a.ptr[s];
  const int len = a.len[s * kRowsA + lane];
  y[0] = y[1] = y[2] = 0.0;
  xo[0] = xo[1] = xo[2] = 0.0;
  if (len == 0) return;
  y[0] = y[1] = y[2] = -0.0;
  const int32_t* __restrict__ colp = a.col + (int64_t)base * kRowsA + lane;
  int k0 = 0;
  for (; k0 + U <= len; k0 += U) sell_chunk<U, true, NT>(a, base, lane, colp, x, k0, len, y, xo);
  if (k0 < len) sell_chunk<U, false, NT>(a, base, lane, colp, x, k0, len, y, xo);
}

// LU solve with the factors of hecmw_precond_SSOR_33.F90:183-195 (inverted
// pivots on the diagonal, multipliers below): the reference's statements.
template <typename T>
__device__ __forceinline__ void lu3_solve(const T (&a)[9], T& x0, T& x1, T& x2) {
#pragma clang fp contract(off)
  x1 = x1 - a[3] * x0;
  x2 = x2 - a[6] * x0 - a[7] * x1;
  x2 = a[8] * x2;
  x1 = a[4] * (x1 - a[5] * x2);
  x0 = a[0] * (x0 - a[2] * x2 - a[1] * x1);
}

}  // namespace hecmw33
