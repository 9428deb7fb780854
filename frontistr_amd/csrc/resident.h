// Device code that the resident kernels share: exchange between workgroups that all
// stay on the GPU, their grid barrier and their reductions.
#pragma once
#include <hip/hip_runtime.h>

#include <cstdint>

#include "device.h"
#include "rows.h"

namespace hecmw33 {

constexpr int32_t kErrNoconv = 3001;
constexpr int32_t kErrDivergeMat = 3002;
constexpr int32_t kErrDivergePc = 3003;
constexpr int32_t kErrDivergeNan = 3004;

// How the waves exchange vectors: between workgroups every exchanged value is
// written and read at agent scope (sc1: past the caches that other XCDs do not
// see); a single workgroup keeps the gathered vectors in LDS.
enum Exchange : int { kOneGroup = 0, kGrid = 1 };

constexpr uint64_t kWaitTicks = 20ull * 100000000ull;  // 20 s of the 100 MHz wall clock

template <int MEM>
__device__ __forceinline__ double ld(const double* p) {
  if (MEM == kGrid) return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  return *p;
}
template <int MEM>
__device__ __forceinline__ void st(double* p, double v) {
  if (MEM == kGrid)
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  else
    *p = v;
}

// barrier of the workgroup that orders LDS but leaves global loads in flight
// (__syncthreads would wait for the prefetched matrix data)
__device__ __forceinline__ void wg_barrier() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
}
// this wave's stores have completed
__device__ __forceinline__ void drain_stores() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); }
// orders a wave's own LDS accesses (the LDS serves a wave in order)
__device__ __forceinline__ void lds_order() { __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront"); }

// what the workgroups share in `sync`: an abort flag in lines of its own, and from word
// kSyncParts on three sets of two entries per workgroup for the exchanges
constexpr int kSyncParts = 64;
constexpr int kSyncSet = 2 * kResidentGridMax;
static_assert(kResidentSync == kSyncParts + 3 * 2 * kSyncSet, "words of the exchange");

constexpr int kAuxSc1 = 16;  // agent scope, as the cache bits of a buffer access

// The mark of an entry that has not been computed: a quiet NaN with a payload
// that no computed value keeps (unmarked replaces it by the plain NaN).
constexpr int kMarkHi = 0x7FFADEAD;
__device__ __forceinline__ double mark() { return __hiloint2double(kMarkHi, 0); }
__host__ __device__ __forceinline__ bool marked(double v) { return (int)(__builtin_bit_cast(uint64_t, v) >> 32) == kMarkHi; }
__device__ __forceinline__ double unmarked(double v) {
  return marked(v) ? __hiloint2double(0x7FF80000, 0) : v;
}

// The copy of the ring whose first gather is preceded by dropping the caches' lines, of all
// copies.  A copy's old lines must be gone before it is gathered again, so none of them may
// come back between the drop and the marks' return: the copy before this one gets its marks
// right after the drop, and a BiCGSTAB sweep of s^ reads p^ in the copy that it marks.  The
// sweeps of s^ take the even copies (the first sweep of p^ takes copy 1, a refresh takes the
// copy of the sweep that follows it), so the line is drawn at an odd one.
__host__ __device__ __forceinline__ bool drops_lines(int copy) { return copy == 1; }

// Whether a gathered record has to be asked for again: {z} of a backward sweep, {z w} of a
// forward one, where w is what the sweep computes.  z stands in memory by then, but the
// record comes in several loads, and one that the caches serve may bring marks of z from a
// line of the backward sweep beside a w that has just arrived: unless the sweep leaves z
// aside (the refresh, before there is one), every entry counts.  Past the caches z needs no
// look (with_z false): 343 nodes in one workgroup 4.39 ms a solve against 4.54.
template <int NG>
__host__ __device__ __forceinline__ bool missing(const double (&x)[3 * NG], bool with_z) {
  bool m = marked(x[3 * NG - 3]) | marked(x[3 * NG - 2]) | marked(x[3 * NG - 1]);
  if (NG > 1 && with_z) m |= marked(x[0]) | marked(x[1]) | marked(x[2]);
  return m;
}

// The LDS that a resident kernel may ask for.  A kernel's attributes belong to the process, so
// every launch of any context sets this one value, whatever its own size is.
inline hipError_t allow_lds(const void* kernel) {
  return hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, kLdsBytes);
}

template <int J>
__device__ __forceinline__ double quad_bcast(double v) {
  constexpr int ctrl = J | (J << 2) | (J << 4) | (J << 6);
  const int lo = __builtin_amdgcn_mov_dpp(__double2loint(v), ctrl, 0xf, 0xf, false);
  const int hi = __builtin_amdgcn_mov_dpp(__double2hiint(v), ctrl, 0xf, 0xf, false);
  return __hiloint2double(hi, lo);
}

// by one workgroup, before a launch
__device__ __forceinline__ void reset_sync(uint32_t* sync) {
  for (int i = threadIdx.x; i < kSyncParts; i += blockDim.x) sync[i] = 0;
  double* const parts = reinterpret_cast<double*>(sync + kSyncParts);
  for (int i = threadIdx.x; i < 3 * kSyncSet; i += blockDim.x) parts[i] = mark();
}

// A workgroup of T threads in the grid
template <int T, int MEM>
struct GridGroup {
  static constexpr int kWaves = T / kWave;
  static constexpr int kRedDoubles = 2 * kWaves + 8;  // LDS at `red`

  uint32_t* sync;
  double* red;
  int lane, wave, G, blk;
  int set = 0;         // of the next exchange
  bool dead = false;   // a wait ran out (this wave's view): go on without waiting

  __device__ __forceinline__ GridGroup(uint32_t* counters, double* scratch) : sync(counters), red(scratch) {
    lane = threadIdx.x & (kWave - 1);
    wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    G = gridDim.x;
    blk = xcd_block(blockIdx.x, G);
  }

  // a wait that has run long: whether to give it up
  __device__ __forceinline__ bool give_up(uint64_t& t0) {
    const uint64_t now = wall_clock64();
    if (t0 == 0) t0 = now;
    if (now - t0 > kWaitTicks) __hip_atomic_store(sync, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    return __hip_atomic_load(sync, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0;
  }

  // Sums of K2 values per workgroup (lane k < K2 of wave 0 brings value k) by wave 0, the
  // same everywhere, and the grid barrier: the workgroups read each other's entries, again
  // while one still holds its mark, so that the chain is one store and one load.
  // Three sets of entries take turns: everyone has read the set before once all have
  // written this one, so this workgroup's entries there get their marks back
  // then, and the next exchange but one uses them.
  // CG with diagonal scaling, two exchanges an iteration: with arrival counters and the
  // entries read after them 7.2 us at 4 workgroups, 8.2 at 35, 10.1 at 145, 15.0 at 256; this
  // way 6.1, 7.0, 8.6 and 14.8.  (Two stages of 16 entries: no better than the counters.)
  template <int K2>
  __device__ __forceinline__ void exchange(double own, double (&tot)[K2]) {
    constexpr int kPer = kResidentGridMax / kWave;
    double* const parts = reinterpret_cast<double*>(sync + kSyncParts);
    double* const at = parts + set * kSyncSet;
    double u[K2][kPer];
    drain_stores();
    if (lane < K2) st<kGrid>(at + lane * kResidentGridMax + blk, unmarked(own));
#pragma unroll
    for (int k = 0; k < K2; ++k)
#pragma unroll
      for (int q = 0; q < kPer; ++q) u[k][q] = lane + q * kWave < G ? mark() : 0.0;
    uint64_t t0 = 0;
    for (uint32_t spins = 1; !dead; ++spins) {
      bool more = false;
#pragma unroll
      for (int k = 0; k < K2; ++k)
#pragma unroll
        for (int q = 0; q < kPer; ++q)
          if (marked(u[k][q])) u[k][q] = ld<kGrid>(at + k * kResidentGridMax + lane + q * kWave);
#pragma unroll
      for (int k = 0; k < K2; ++k)
#pragma unroll
        for (int q = 0; q < kPer; ++q) more |= marked(u[k][q]);
      if (!__any(more)) break;
      if ((spins & 1023u) == 0) dead = __any(lane == 0 && give_up(t0));
    }
#pragma unroll
    for (int k = 0; k < K2; ++k) {
      double t = u[k][0];
#pragma unroll
      for (int q = 1; q < kPer; ++q) t += u[k][q];
      tot[k] = wave_sum(t);
    }
    if (lane < 2) st<kGrid>(parts + (set == 0 ? 2 : set - 1) * kSyncSet + lane * kResidentGridMax + blk, mark());
    set = set == 2 ? 0 : set + 1;
  }
  // grid barrier for stores that the callers have drained
  __device__ __forceinline__ void grid_sync() {
    wg_barrier();
    if (MEM == kOneGroup) return;
    if (wave == 0) {
      double t[1];
      exchange<1>(0.0, t);
    }
    wg_barrier();
  }
  // barrier for plain stores too: x in node order, which the product reads
  // through the caches
  __device__ __forceinline__ void full_sync() {
    drain_stores();
    wg_barrier();
    if (MEM == kOneGroup) return;
    if (wave == 0) {
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "agent");
      double t[1];
      exchange<1>(0.0, t);
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
    }
    wg_barrier();
  }

  // totals of K2 per-lane sums over the grid, the same on every thread: a wave
  // tree, the workgroup's waves in order, then a fixed tree over the
  // workgroups.  Also a grid barrier, for stores that the callers have drained.
  template <int K2>
  __device__ __forceinline__ void reduce(const double (&in)[K2], double (&tot)[K2]) {
#pragma unroll
    for (int k = 0; k < K2; ++k) {
      const double w = wave_sum(in[k]);
      if (lane == 0) red[k * kWaves + wave] = w;
    }
    wg_barrier();
    if (wave == 0) {
      double s = 0.0;
      if (lane < K2) {
        s = red[lane * kWaves];
        for (int w = 1; w < kWaves; ++w) s += red[lane * kWaves + w];
      }
      if (MEM == kGrid) {
        double t[K2];
        exchange<K2>(s, t);
#pragma unroll
        for (int k = 0; k < K2; ++k)
          if (lane == 0) red[2 * kWaves + k] = t[k];
      } else if (lane < K2) {
        red[2 * kWaves + lane] = s;
      }
    }
    wg_barrier();
#pragma unroll
    for (int k = 0; k < K2; ++k) tot[k] = red[2 * kWaves + k];
    wg_barrier();
  }
};

}  // namespace hecmw33
