// The FP32 SSOR application of the flexible CG as one kernel: the colour launches'
// statements in the same order, the colours following each other as a dataflow.
//
// A launch per colour takes 5-7 us whatever its size up to 10,000 rows (launch gap, then
// row -> column -> gather -> next chunk from a cold L2), 33 of them 0.2 ms, while the
// matrix stream of a 48^3 cube alone would take 12 us.  Here
//  * a wave works on a slice of 16 rows, four lanes per row, and loads its next
//    slice's matrix data before it waits for anything;
//  * a row's result is a 16-byte record; one that is not there yet holds marked NaNs
//    and is read again until it is;
//  * workgroups draw their slices, eight at a time in the order of the sweeps, from a
//    counter: whoever waits does so for slices drawn before its own, so the kernel
//    ends however few of its workgroups are on the GPU, and an ordinary launch does
//    (a cooperative one costs 20 us).
// The values are packed so that a lane finds those of eight blocks in three 16-byte
// loads (BF16; six in FP32) instead of 24 two-byte ones, and the four lanes of a row
// gather a block each instead of one entry of all.
// Measured, us per application with BF16 values, launch per colour -> this (HEX8 cubes):
// 27 nodes 100 -> 51, 9,261 163 -> 95, 29,791 160 -> 92, 117,649 184 -> 100, 226,981 207 ->
// 116, 389,017 282 -> 171, 1,030,301 510 -> 343; in FP32 206 -> 131 and 284 -> 200 at 226,981
// and 389,017.  Up to 100,000 nodes the 2 x 16 colour steps bound it, 2.4 us each (a
// store's way to memory, the gather's way back, the row's ordered sum), above
// that the gathers past the caches.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>

#include "device.h"
#include "resident.h"
#include "rows.h"

namespace hecmw33 {
namespace {

constexpr int kFlowThreads = 512;
constexpr int kFlowWaves = kFlowThreads / kWave;
constexpr int kFlowGroups = 2;  // groups of kFlowBlocks blocks of a row that are loaded ahead

using U4 = __attribute__((__vector_size__(16))) uint32_t;

// marked entries, as in the FP64 kernels
constexpr uint32_t kMark32 = 0x7FFADEADu;
__device__ __forceinline__ uint32_t unmarked32(float v) {
  const uint32_t u = __float_as_uint(v);
  return u == kMark32 ? 0x7FC00000u : u;
}
template <int J>
__device__ __forceinline__ float quad_bcast32(float v) {
  return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), J | J << 2 | J << 4 | J << 6, 0xf, 0xf, false));
}

// value 3 j + e of a lane's group: packed BF16 pairs, or FP32
template <bool B16>
struct Values {
  static constexpr int kPlanes = B16 ? 3 : 6;  // of 48 lanes x 16 bytes
  U4 p[kPlanes];
  __device__ __forceinline__ void load(const U4* __restrict__ v, int64_t g, int l48) {
#pragma unroll
    for (int i = 0; i < kPlanes; ++i) p[i] = v[(g * kPlanes + i) * 48 + l48];
  }
  __device__ __forceinline__ float get(int idx) const {
    if (B16) {
      const uint32_t w = p[idx / 8][idx % 8 / 2];
      return __uint_as_float(idx % 2 ? w & 0xffff0000u : w << 16);
    }
    return __uint_as_float(p[idx / 4][idx % 4]);
  }
};

template <bool B16>
struct Flow {
  const FlowOp& o;
  __amdgpu_buffer_rsrc_t rec;  // records of the forward, then of the backward result
  int lane, r, d, dd, l48;
  bool dead = false;
  // the wave's next slice
  int dir, s, ng, len;
  int32_t node;
  int2 col[kFlowGroups];
  Values<B16> val[kFlowGroups];
  float a[9];
  float4 rhs;

  __device__ __forceinline__ explicit Flow(const FlowOp& op) : o(op) {
    rec = __builtin_amdgcn_make_buffer_rsrc(o.rec, 0, (int)(uint32_t)(32 * (int64_t)o.ns), 0x00020000);
    lane = threadIdx.x & (kWave - 1);
    r = lane >> 2;
    d = lane & 3;
    dd = d < 3 ? d : 2;
    l48 = 3 * r + dd;
  }
  __device__ __forceinline__ void load_group(int g, int2& c, Values<B16>& v) const {
    const int64_t at = (int64_t)o.group[dir][s] + g;
    c = o.col[dir][at * kWave + lane];
    v.load(reinterpret_cast<const U4*>(o.val[dir]), at, l48);
  }
  // task t of both sweeps: the slices forward, then backward
  __device__ __forceinline__ void load(int64_t t) {
    const int S = o.ns / kRowsS;
    dir = t < S ? 0 : 1;
    s = (int)(dir ? 2 * (int64_t)S - 1 - t : t);
    if (s < 0) return;
    const int slot = s * kRowsS + r;
    ng = o.group[dir][s + 1] - o.group[dir][s];
#pragma unroll
    for (int g = 0; g < kFlowGroups; ++g)
      if (g < ng) load_group(g, col[g], val[g]);
    len = o.len[dir][slot];
    node = o.row_old[slot];
    const float* f = o.alu + (int64_t)s * 9 * kRowsS + r;
#pragma unroll
    for (int e = 0; e < 9; ++e) a[e] = f[e * kRowsS];
    if (!dir) rhs = o.rhs[slot];
  }
  __device__ __forceinline__ bool fetch(uint32_t at, float (&x)[3]) const {
    const U4 v = __builtin_amdgcn_raw_buffer_load_b128(rec, at * 16, 0, kAuxSc1);
    x[0] = __uint_as_float(v[0]);
    x[1] = __uint_as_float(v[1]);
    x[2] = __uint_as_float(v[2]);
    return v[0] == kMark32 || v[1] == kMark32 || v[2] == kMark32;
  }
  // the records of N groups' blocks (this lane's: d and d + 4 of each), and with `own`
  // the row's own, once they are there
  template <int N>
  __device__ __forceinline__ void gather(const int2 (&c)[N], int g0, bool with_own, float (&x)[2 * N][3], float (&own)[3]) {
    bool want[2 * N], want_own = with_own && node >= 0;
#pragma unroll
    for (int g = 0; g < N; ++g) {
      want[2 * g] = (g0 + g) * kFlowBlocks + d < len;
      want[2 * g + 1] = (g0 + g) * kFlowBlocks + 4 + d < len;
    }
    const uint32_t base = dir ? o.ns : 0;
    uint64_t t0 = 0;
    for (uint32_t spins = 1;; ++spins) {
      bool more = false;
#pragma unroll
      for (int g = 0; g < N; ++g) {
        if (want[2 * g]) want[2 * g] = fetch(base + c[g].x, x[2 * g]);
        if (want[2 * g + 1]) want[2 * g + 1] = fetch(base + c[g].y, x[2 * g + 1]);
      }
      if (want_own) want_own = fetch(s * kRowsS + r, own);
#pragma unroll
      for (int i = 0; i < 2 * N; ++i) more |= want[i];
      if (!__any(more || want_own) || dead) break;
      if ((spins & 1023u) == 0) {
        // a wait that has run long is given up: marks, which are NaN, go on, and at the end
        // the host is told
        const uint64_t now = wall_clock64();
        if (t0 == 0) t0 = now;
        dead = __any(now - t0 > kWaitTicks);
      }
    }
  }
  __device__ __forceinline__ void add(const Values<B16>& v, const float (&x0)[3], const float (&x1)[3], int g, float& sw) const {
#pragma clang fp contract(off)
    auto block = [&](int j, float b0, float b1, float b2) {
      const float v0 = v.get(3 * j), v1 = v.get(3 * j + 1), v2 = v.get(3 * j + 2);
      const float t = dir ? sw + v0 * b0 + v1 * b1 + v2 * b2 : sw - v0 * b0 - v1 * b1 - v2 * b2;
      sw = g * kFlowBlocks + j < len ? t : sw;
    };
    block(0, quad_bcast32<0>(x0[0]), quad_bcast32<0>(x0[1]), quad_bcast32<0>(x0[2]));
    block(1, quad_bcast32<1>(x0[0]), quad_bcast32<1>(x0[1]), quad_bcast32<1>(x0[2]));
    block(2, quad_bcast32<2>(x0[0]), quad_bcast32<2>(x0[1]), quad_bcast32<2>(x0[2]));
    block(3, quad_bcast32<3>(x0[0]), quad_bcast32<3>(x0[1]), quad_bcast32<3>(x0[2]));
    block(4, quad_bcast32<0>(x1[0]), quad_bcast32<0>(x1[1]), quad_bcast32<0>(x1[2]));
    block(5, quad_bcast32<1>(x1[0]), quad_bcast32<1>(x1[1]), quad_bcast32<1>(x1[2]));
    block(6, quad_bcast32<2>(x1[0]), quad_bcast32<2>(x1[1]), quad_bcast32<2>(x1[2]));
    block(7, quad_bcast32<3>(x1[0]), quad_bcast32<3>(x1[1]), quad_bcast32<3>(x1[2]));
  }
  __device__ __forceinline__ void work() {
#pragma clang fp contract(off)
    float x[2 * kFlowGroups][3], own[3] = {0.f, 0.f, 0.f};
    gather<kFlowGroups>(col, 0, dir != 0, x, own);
    float sw = dir ? 0.f : (dd == 0 ? rhs.x : (dd == 1 ? rhs.y : rhs.z));
#pragma unroll
    for (int g = 0; g < kFlowGroups; ++g)
      if (g < ng) add(val[g], x[2 * g], x[2 * g + 1], g, sw);
#pragma unroll 1
    for (int g = kFlowGroups; g < ng; ++g) {
      int2 c[1];
      Values<B16> v;
      float y[2][3], none[3];
      load_group(g, c[0], v);
      gather<1>(c, g, false, y, none);
      add(v, y[0], y[1], g, sw);
    }
    float x0 = quad_bcast32<0>(sw), x1 = quad_bcast32<1>(sw), x2 = quad_bcast32<2>(sw);
    lu3_solve<float>(a, x0, x1, x2);
    if (dir) {
      x0 = own[0] - x0;
      x1 = own[1] - x1;
      x2 = own[2] - x2;
    }
    if (node >= 0 && d == 0) {
      const U4 w = {unmarked32(x0), unmarked32(x1), unmarked32(x2), 0u};
      __builtin_amdgcn_raw_buffer_store_b128(w, rec, (uint32_t)((dir ? o.ns : 0) + s * kRowsS + r) * 16, 0, kAuxSc1);
    }
  }
};

template <bool B16>
__global__ __launch_bounds__(kFlowThreads) void k_ssor_flow(FlowOp o, const KrylovState* st) {
  if (st && st->done) return;
  __shared__ uint32_t drawn[2];
  Flow<B16> f(o);
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const uint32_t ntask = 2 * (uint32_t)(o.ns / kRowsS), end = (ntask + kFlowWaves - 1) / kFlowWaves;
  auto draw = [&] { return __hip_atomic_fetch_add(o.ticket, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); };
  if (threadIdx.x == 0) drawn[0] = draw();
  wg_barrier();
  uint32_t now = drawn[0], task = now * kFlowWaves + wave;
  if (task < ntask) f.load(task);
  for (int turn = 1; now < end; turn ^= 1) {
    uint32_t t = 0;
    if (threadIdx.x == 0) t = draw();
    if (task < ntask) f.work();
    if (threadIdx.x == 0) drawn[turn] = t;
    wg_barrier();
    now = drawn[turn];
    task = now * kFlowWaves + wave;
    if (task < ntask) f.load(task);
  }
  if (f.dead && f.lane == 0) __hip_atomic_store(o.gave_up, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

// r into slot order, the records marked, the counter at zero
__global__ __launch_bounds__(kBlock) void k_flow_stage(FlowOp o, const float* __restrict__ r, const KrylovState* st) {
  if (st && st->done) return;
  if (blockIdx.x == 0 && threadIdx.x == 0) *o.ticket = 0;
  const float m = __uint_as_float(kMark32);
  for (int64_t t = (int64_t)blockIdx.x * kBlock + threadIdx.x; t < o.ns; t += (int64_t)gridDim.x * kBlock) {
    const int64_t i = o.row_old[t];
    float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
    if (i >= 0) v = make_float4(r[3 * i], r[3 * i + 1], r[3 * i + 2], 0.f);
    o.rhs[t] = v;
    const float4 mk = make_float4(m, m, m, 0.f);
    reinterpret_cast<float4*>(o.rec)[t] = mk;
    reinterpret_cast<float4*>(o.rec)[o.ns + t] = mk;
  }
}

// FP64 values of a SELL-16 factor -> FP32 -> (BF16, round to nearest even) in the packed
// layout, and with `col` its columns; backward rows from their last block on
template <bool B16>
__global__ __launch_bounds__(kBlock) void k_flow_pack(Sell<double> m, const int32_t* __restrict__ group, int desc,
                                                       U4* __restrict__ val, int2* __restrict__ col) {
  constexpr int kPer = B16 ? 8 : 4, kPlanes = Values<B16>::kPlanes;
  const int lane = threadIdx.x & (kWave - 1);
  for (int s = blockIdx.x * (kBlock / kWave) + threadIdx.x / kWave; s < m.nslices; s += gridDim.x * (kBlock / kWave)) {
    const int64_t base = m.ptr[s];
    for (int64_t g = group[s]; g < group[s + 1]; ++g) {
      const int b0 = (int)(g - group[s]) * kFlowBlocks;
      if (lane < 48) {
        const int r = lane / 3, dd = lane % 3, len = m.len[s * kRowsS + r];
        for (int i = 0; i < kPlanes; ++i) {
          uint32_t w[kPer];
          for (int q = 0; q < kPer; ++q) {
            const int idx = i * kPer + q, k = b0 + idx / 3, kk = desc ? len - 1 - k : k;
            w[q] = 0;
            if (k < len) {
              w[q] = __float_as_uint((float)m.val[((base + kk) * 9 + 3 * dd + idx % 3) * kRowsS + r]);
              if (B16) w[q] = (w[q] + 0x7FFFu + ((w[q] >> 16) & 1u)) >> 16;
            }
          }
          U4 p;
          for (int q = 0; q < 4; ++q) p[q] = B16 ? w[2 * q % kPer] | w[(2 * q + 1) % kPer] << 16 : w[q % kPer];
          val[(g * kPlanes + i) * 48 + lane] = p;
        }
      }
      if (col) {
        const int r = lane >> 2, len = m.len[s * kRowsS + r];
        int c[2];
        for (int h = 0; h < 2; ++h) {
          const int k = b0 + 4 * h + (lane & 3), kk = desc ? len - 1 - k : k;
          c[h] = k < len ? m.col[(base + kk) * kRowsS + r] : 0;
        }
        col[g * kWave + lane] = make_int2(c[0], c[1]);
      }
    }
  }
}

}  // namespace

void flow_pack(const Sell<double>& m, const int32_t* group, bool desc, bool b16, void* val, int2* col, hipStream_t s) {
  const int g = std::min(std::max((m.nslices + kBlock / kWave - 1) / (kBlock / kWave), 1), 8192);
  if (b16)
    k_flow_pack<true><<<g, kBlock, 0, s>>>(m, group, desc ? 1 : 0, static_cast<U4*>(val), col);
  else
    k_flow_pack<false><<<g, kBlock, 0, s>>>(m, group, desc ? 1 : 0, static_cast<U4*>(val), col);
}

void flow_sweeps(const FlowOp& o, const float* r, const KrylovState* st, hipStream_t s) {
  k_flow_stage<<<std::min(std::max((o.ns + kBlock - 1) / kBlock, 1), 2048), kBlock, 0, s>>>(o, r, st);
  if (o.b16)
    k_ssor_flow<true><<<o.grid, kFlowThreads, 0, s>>>(o, st);
  else
    k_ssor_flow<false><<<o.grid, kFlowThreads, 0, s>>>(o, st);
}

}  // namespace hecmw33
