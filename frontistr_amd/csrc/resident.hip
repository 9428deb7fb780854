// SSOR-CG and SSOR-BiCGSTAB as one resident kernel: every workgroup stays on the
// GPU for many iterations.
//
// What bounds the launch-per-colour solve below about a million rows is not the
// matrix stream but the chain of ~35 dependent launches per SSOR application
// (5-11 us each: launch gap, then row length -> column -> gather -> next chunk
// from a cold L2).  Here the sweeps run as a dataflow between waves:
//  * The blocks of up to 16 consecutive rows of a colour form a task of 64 lanes
//    x K blocks, a row taking whole lanes, so that a wave needs one round of
//    loads per task whatever the rows' lengths are.  A workgroup's tasks go
//    round robin over its waves in the order of the sweep; a wave loads its next
//    task's matrix data while it works on the present one.
//  * A gathered entry that is not there yet is a marked NaN, and the wave loads
//    it again until it is: no barrier between colours, no flag, no store to be
//    waited for.  (With grid barriers between the colours a step cost 3.7 us at
//    9,261 nodes, 2.2 us of them the barrier.)
//  * Every entry is written once per sweep.  Copies take turns, and a backward
//    sweep puts the marks back into the copy that the sweep before used; the
//    reductions between the sweeps are grid barriers.  With four copies (from 17,000 nodes
//    on) the first look at an entry goes through the caches (a record is gathered about 13 times in
//    a sweep, and past the caches that was half of the memory traffic at 72^3); an
//    old line can only hold marks, because the lines go once per turn of the copies, and
//    a record with a mark in any entry that the sweep uses is asked for again past the
//    caches.
//
// The iteration needs the off-diagonal blocks once, not twice as SSOR
// application + product do.  With A = L + D + U and M = (D'+L) D'^-1 (D'+U)
// (D' = D with sigma on its diagonal), u = (D'+L)^-1 r and z = M^-1 r satisfy
// (D'+U) z = D' u, hence A z = L z + D' u + (D - D') z, and the forward sweep
// for w = (D'+L)^-1 A z meets every L block with both z_j and w_j.  (Eisenstat's
// observation, SIAM J. Sci. Stat. Comput. 2 (1981) 1-4, with the residual kept
// beside its transformed form, because the convergence test reads |r|.)  The
// vectors carried in slot order, D'-multiplied so that no row needs D':
//   h = D' u, t = A z - L w = D' w, p = z + beta p, q = A p = A z + beta q,
//   g = D' (D'+L)^-1 q = t + beta g
//   backward (colours descending): h -= alpha g, r -= alpha q, x += alpha p,
//     z = D'^-1 (h - U z); partials r.r, r.z
//   forward (ascending): A z = L z + h + (D - D') z, t = A z - L w, w = D'^-1 t,
//     p, q, g; partial p.q
// Measured, us per iteration, launches per colour -> resident (HEX8 cubes and a
// TET10 box, relative residual 1e-10): 343 nodes 183 -> 47, 4,845 (TET10) 441 ->
// 80, 9,261 298 -> 64, 29,791 289 -> 65, 74,088 376 -> 81, 389,017 717 -> 288,
// 1,030,301 1400 -> 774.  Up to 100,000 nodes the 2 x 16 colour steps bound it
// (1.5-2 us each: gather round trip, row work, the way of the stores to the
// neighbours' gathers); above, the round trips of a wave's tasks (8 waves per CU; the
// matrix stream alone would take 200 us at 389,017).
//
// The true residual b - A x (every 50 iterations and before convergence is
// declared, as the reference does) is formed in natural order with the rows of
// the plain SpMV, and h and z are then rebuilt from it by plain sweeps.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>
#include <type_traits>

#include "device.h"
#include "resident.h"
#include "rows.h"

namespace hecmw33 {
namespace {

// The gathered vectors z and w of a row share a record {z0 z1 z2 w0 w1 w2}, of 64
// bytes in memory, read with 16-byte loads: three requests for both vectors,
// two for z alone, instead of one per entry.  Buffer loads, because only they
// take 16 bytes with the agent-scope bit.
using V4 = __attribute__((__vector_size__(16))) uint32_t;
using V2 = __attribute__((__vector_size__(8))) uint32_t;
template <int AUX>
__device__ __forceinline__ void gather16(__amdgpu_buffer_rsrc_t r, uint32_t off, double& a, double& b) {
  const V4 v = __builtin_amdgcn_raw_buffer_load_b128(r, off, 0, AUX);
  a = __hiloint2double((int)v[1], (int)v[0]);
  b = __hiloint2double((int)v[3], (int)v[2]);
}
template <int AUX>
__device__ __forceinline__ double gather8(__amdgpu_buffer_rsrc_t r, uint32_t off) {
  const V2 v = __builtin_amdgcn_raw_buffer_load_b64(r, off, 0, AUX);
  return __hiloint2double((int)v[1], (int)v[0]);
}

// LDS of a workgroup: products (kComp per lane and wave), reduction scratch,
// the count of finished tasks, per direction and colour {first task, tasks
// before it}, and with one workgroup the gathered vectors
constexpr int kComp = 6;
template <int T>
struct LdsMap {
  static constexpr int kWaves = T / kWave;
  static constexpr int prod = 0;
  static constexpr int red = prod + kWaves * kWave * kComp;
  static constexpr int fin = red + 2 * kWaves + 8;
  static constexpr int range = fin + 2;  // in doubles; int2 each
  static size_t bytes(int ncolor, int one_group_slots) {
    return sizeof(double) * (range + 2 * (size_t)(ncolor + 1) + (one_group_slots ? 12 * ((size_t)one_group_slots + 1) : 0));
  }
};

template <int T, int K, int MEM>
struct Resident : GridGroup<T, MEM> {
  using Map = LdsMap<T>;
  using Group = GridGroup<T, MEM>;
  using Group::blk;
  using Group::dead;
  using Group::G;
  using Group::kWaves;
  using Group::lane;
  using Group::wave;
  static constexpr int kRec = MEM == kGrid ? 8 : 6;  // doubles of a gathered record

  const ResidentOp& o;
  __amdgpu_buffer_rsrc_t rsrc;
  double* zw0;           // the copies of the gathered records (o.ring), copy_size doubles each
  int64_t copy_size;
  double* prod;
  uint32_t* fin;
  const int2* range;
  int par = 0;           // copy that holds the present z and w
  uint32_t fin0 = 0;     // tasks finished before this sweep
  // the wave's next task: its place in the workgroup's order of the sweep, its
  // colour step and the tasks before that, its rows and lanes, its matrix data
  int j, step, before;
  int4 desc;
  double v[K][9];
  int32_t c[K];

  __device__ __forceinline__ Resident(const ResidentOp& op, double* lds) : Group(op.sync, lds + Map::red), o(op) {
    prod = lds + Map::prod + wave * kWave * kComp;
    fin = reinterpret_cast<uint32_t*>(lds + Map::fin);
    int2* rg = reinterpret_cast<int2*>(lds + Map::range);
    range = rg;
    const int nc = o.ncolor;
    copy_size = ((int64_t)o.ns + 1) * kRec;
    if (MEM == kGrid) {
      zw0 = o.zw;
      rsrc = __builtin_amdgcn_make_buffer_rsrc(o.zw, 0, (int)(uint32_t)(o.ring * sizeof(double) * copy_size), 0x00020000);
    } else {
      zw0 = lds + Map::range + 2 * (nc + 1);
      // the state of the gathered vectors between launches is in o.zw
      for (int64_t i = threadIdx.x; i < o.ring * copy_size; i += T) zw0[i] = o.zw[i];
    }
    // this workgroup's run of the tasks of every colour, and how many go before
    for (int i = threadIdx.x; i < 2 * (nc + 1); i += T) {
      const int d = i / (nc + 1), k = i - d * (nc + 1);  // k-th step of the sweep
      const int32_t* ct = o.color_task + d * (nc + 1);
      int2 r = make_int2(0, 0);
      for (int q = 0; q < k; ++q) {
        const int cq = d ? nc - 1 - q : q;
        const int64_t n = ct[cq + 1] - ct[cq];
        r.y += (int)(n * (blk + 1) / G) - (int)(n * blk / G);
      }
      if (k < nc) {
        const int ck = d ? nc - 1 - k : k;
        const int64_t n = ct[ck + 1] - ct[ck];
        r.x = ct[ck] + (int)(n * blk / G);
      }
      rg[i] = r;
    }
    if (threadIdx.x == 0) *fin = 0;
    __syncthreads();
  }

  __device__ __forceinline__ int next_copy() const { return par + 1 == o.ring ? 0 : par + 1; }
  __device__ __forceinline__ int last_copy() const { return par == 0 ? o.ring - 1 : par - 1; }
  // The caches may hold lines of a copy from before its marks were put back: between the
  // barrier behind the last gather or mark of that time and the next gather, they go.
  __device__ __forceinline__ void drop_lines() {
    if (MEM == kOneGroup || !o.cached) return;
    if (wave == 0) __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
    wg_barrier();
  }
  // once per turn of the ring, before copy cp is gathered
  __device__ __forceinline__ void enter(int cp) {
    if (drops_lines(cp)) drop_lines();
  }
  __device__ __forceinline__ double* zw(int cp, int slot) const { return zw0 + cp * copy_size + (int64_t)kRec * slot; }

  // The wave's place j in the workgroup's order of the sweep in direction d (0
  // forward, 1 backward): its task (-1: past the end), the step's number and
  // how many tasks go before the step; the step is at least `from`.
  __device__ __forceinline__ int find(int d, int at, int from, int& step_at, int& before) const {
    const int nc = o.ncolor;
    const int2* r = range + d * (nc + 1);
    int2 lo = r[from];
    for (; from < nc; ++from) {
      const int2 hi = r[from + 1];
      if (at < hi.y) break;
      lo = hi;
    }
    step_at = from;
    before = lo.y;
    return from < nc ? lo.x + at - lo.y : -1;
  }
  __device__ __forceinline__ void load(int t) {
    desc = o.task[t];
    const bool used = lane < desc.z;
#pragma unroll
    for (int k = 0; k < K; ++k) {
      const int64_t g = (int64_t)t * K + k;
      c[k] = o.ns;
#pragma unroll
      for (int e = 0; e < 9; ++e) v[k][e] = 0.0;
      if (used) {
        if (o.stream) {
          c[k] = __builtin_nontemporal_load(o.col + g * kWave + lane);
          aval_load_nt(o.val, g, lane, v[k]);
        } else {
          c[k] = o.col[g * kWave + lane];
          aval_load(o.val, g, lane, v[k]);
        }
      }
    }
  }
  // the wave's first task of a sweep
  __device__ __forceinline__ void begin(int d) {
    j = wave;
    const int t = find(d, j, 0, step, before);
    if (t >= 0) load(t);
  }

  // the gathered records of the task's blocks from copy `cp`, again until their
  // entries are there (see missing)
  template <int NG>
  __device__ __forceinline__ void gather(int cp, bool with_z, double (&x)[K][3 * NG]) {
    bool want[K];
#pragma unroll
    for (int k = 0; k < K; ++k) want[k] = true;
    uint64_t t0 = 0;
    auto fetch = [&](int k, auto aux) {
      const uint32_t off = (uint32_t)(cp * copy_size * 8) + (uint32_t)c[k] * (8u * kRec);
      gather16<aux.value>(rsrc, off, x[k][0], x[k][1]);
      if constexpr (NG > 1) {
        gather16<aux.value>(rsrc, off + 16, x[k][2], x[k][3]);
        gather16<aux.value>(rsrc, off + 32, x[k][4], x[k][5]);
      } else {
        x[k][2] = gather8<aux.value>(rsrc, off + 16);
      }
    };
    for (uint32_t spins = 1;; ++spins) {
#pragma unroll
      for (int k = 0; k < K; ++k)
        if (want[k]) {
          if constexpr (MEM == kGrid) {
            if (spins == 1 && o.cached)
              fetch(k, std::integral_constant<int, 0>{});
            else
              fetch(k, std::integral_constant<int, kAuxSc1>{});
          } else {
            const volatile double* q = zw(cp, c[k]);
#pragma unroll
            for (int e = 0; e < 3 * NG; ++e) x[k][e] = q[e];
          }
        }
      bool more = false;
#pragma unroll
      for (int k = 0; k < K; ++k) {
        want[k] = missing<NG>(x[k], with_z);
        more |= want[k];
      }
      if (!__any(more) || dead) break;
      if ((spins & 1023u) == 0) dead = __any(lane == 0 && this->give_up(t0));
    }
  }

  // One sweep in direction d over copy `cp` of the gathered records, NG vectors
  // gathered, row work by f; `begin` has been called for it, and is called for
  // the sweep in the other direction at the end.  Row work takes four lanes
  // per row (lane 4 r + e: entry e, the fourth mirrors the third).  with_z: f uses
  // the sums over the gathered z (a refresh has none yet).
  template <int NG, class F>
  __device__ __forceinline__ void sweep(int d, int cp, F& f, bool with_z = true) {
    const int2* r = range + d * (o.ncolor + 1);
    const int total = r[o.ncolor].y;
    const int e = (lane & 3) < 3 ? lane & 3 : 2, row = lane >> 2;
#pragma unroll 1
    while (j < total) {
      const int row0 = desc.x, nr = desc.y;
      const int slot = row0 + min(row, nr - 1);
      const int2 info = o.row[(int64_t)d * o.ns + slot];
      f.pre(slot, e);
      // the task after this one: in this sweep, or the first of the next
      const uint32_t first = fin0 + (uint32_t)before;
      j += kWaves;
      int next = find(d, j, step, step, before);
      if (next < 0) {
        int first_step, first_before;
        next = find(1 - d, wave, 0, first_step, first_before);
      }
      // Look at the neighbours' entries when this workgroup's own tasks of the
      // steps before are finished: the others are about as far, and a wave
      // that asks earlier only loads the memory.
      while ((int32_t)(__hip_atomic_load(fin, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP) - first) < 0)
        __builtin_amdgcn_s_sleep(1);
      double x[K][3 * NG];
      gather<NG>(cp, MEM == kGrid && o.cached && with_z, x);
#pragma unroll
      for (int g = 0; g < NG; ++g)
#pragma unroll
        for (int i = 0; i < 3; ++i) {
          double s = v[0][3 * i] * x[0][3 * g];
          s = fma(v[0][3 * i + 2], x[0][3 * g + 2], fma(v[0][3 * i + 1], x[0][3 * g + 1], s));
#pragma unroll
          for (int k = 1; k < K; ++k)
            s = fma(v[k][3 * i + 2], x[k][3 * g + 2], fma(v[k][3 * i + 1], x[k][3 * g + 1], fma(v[k][3 * i], x[k][3 * g], s)));
          prod[(3 * g + i) * kWave + lane] = s;
        }
      lds_order();
      if (row < nr) {
        const double* pr = prod + e * kWave + (info.x & (kWave - 1));
        const int len = info.y;
        double s[NG] = {};
#pragma unroll 1
        for (int k = 0; k < len; k += 4) {
          double y[NG][4];
#pragma unroll
          for (int u = 0; u < 4; ++u)
#pragma unroll
            for (int g = 0; g < NG; ++g) y[g][u] = pr[3 * g * kWave + min(k + u, len - 1)];
#pragma unroll
          for (int u = 0; u < 4; ++u)
#pragma unroll
            for (int g = 0; g < NG; ++g) s[g] += k + u < len ? y[g][u] : 0.0;
        }
        f.post(slot, e, (lane & 3) < 3, s);
      }
      lds_order();
      if (lane == 0) __hip_atomic_fetch_add(fin, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
      // after the stores: others wait for those
      if (next >= 0) load(next);
    }
    if (total <= wave) begin(1 - d);  // no task of this sweep was this wave's
    j = wave;
    find(1 - d, j, 0, step, before);
    fin0 += (uint32_t)total;
    drain_stores();
  }
};

// Row work of the sweeps, one entry of a row per lane.  The LU of a row's D' and
// its vectors sit in one record per 16 slots (plane = 16 slots, o.planes
// planes), so that a lane reaches all of them from one address.
enum Vec : int {
  kAlu = 0, kR = 9, kX = 12,                                // both methods
  kP = 15, kQ = 18, kG = 21, kH = 24, kCgPlanes = 27,       // CG
  kRt = 15, kBp = 18, kV = 21, kT = 24, kHr = 27, kHp = 30, kHv = 33, kHt = 36, kBiPlanes = 39,  // BiCGSTAB
};
static_assert(kCgPlanes == kResidentPlanesCg && kBiPlanes == kResidentPlanesBi, "planes of a row record");
__device__ __forceinline__ double* rec(const ResidentOp& o, int slot) {
  return o.rec + (int64_t)(slot / kRowsS) * (o.planes * kRowsS) + slot % kRowsS;
}
template <class R, int MEM>
struct Row {
  const R& k;
  double* base;  // entry e of the row's first vector
  double a[9];
  __device__ __forceinline__ explicit Row(const R& res) : k(res) {}
  __device__ __forceinline__ double get(int v) const { return ld<MEM>(base + v * kRowsS); }
  __device__ __forceinline__ void put(int v, double y) const { st<MEM>(base + v * kRowsS, y); }
  __device__ __forceinline__ void begin(int slot, int e) {
    double* b = rec(k.o, slot);
    base = b + e * kRowsS;
#pragma unroll
    for (int i = 0; i < 9; ++i) a[i] = b[(kAlu + i) * kRowsS];
  }
  // entry e of D'^-1 y, y spread over the row's lanes
  __device__ __forceinline__ double solve(double y, int e) const {
    double y0 = quad_bcast<0>(y), y1 = quad_bcast<1>(y), y2 = quad_bcast<2>(y);
    lu3_solve<double>(a, y0, y1, y2);
    return e == 0 ? y0 : (e == 1 ? y1 : y2);
  }
  // the gathered record of a row: z at + e, w at + 3 + e
  __device__ __forceinline__ double* zw(int cp, int slot) const { return k.zw(cp, slot); }
  __device__ __forceinline__ void put_zw(double* p, double y) const {
    if (MEM == kGrid)
      st<MEM>(p, y);
    else
      *const_cast<volatile double*>(p) = y;
  }
};

// CG backward row; upd: with the update of the iteration that ended.  z goes to
// the present copy; the other copy gets its marks back, and after a refresh
// (whose w is in the present copy) so does w.
template <class R, int MEM>
struct RowCgBack : Row<R, MEM> {
  double alpha;
  bool upd;
  double acc[2] = {0.0, 0.0};  // r.r, r.z
  double h, r, g, q, p, x;
  __device__ __forceinline__ RowCgBack(const R& res, double al, bool u) : Row<R, MEM>(res), alpha(al), upd(u) {}
  __device__ __forceinline__ void pre(int slot, int e) {
    this->begin(slot, e);
    h = this->get(kH);
    r = this->get(kR);
    if (upd) {
      g = this->get(kG);
      q = this->get(kQ);
      p = this->get(kP);
      x = this->get(kX);
    }
  }
  __device__ __forceinline__ void post(int slot, int e, bool writes, const double (&s)[1]) {
    if (upd) {
      h = h - alpha * g;
      r = r - alpha * q;
      x = x + alpha * p;
    }
    const double z = this->solve(h - s[0], e);
    if (!writes) return;
    double* now = this->zw(this->k.par, slot) + e;
    double* old = this->zw(this->k.last_copy(), slot) + e;
    this->put_zw(now, unmarked(z));
    this->put_zw(old, mark());
    this->put_zw(old + 3, mark());
    if (upd) {
      this->put(kH, h);
      this->put(kR, r);
      this->put(kX, x);
    } else {
      this->put_zw(now + 3, mark());
    }
    acc[0] += r * r;
    acc[1] += r * z;
  }
};

// CG forward row; refresh: only h and u from r (h = r - L u, w = u), in the copy
// that the next backward sweep takes
template <class R, int MEM>
struct RowCgFwd : Row<R, MEM> {
  double beta;
  bool first, refresh;
  double acc[1] = {0.0};  // p.q
  double h, z, p, q, g, ds;
  __device__ __forceinline__ RowCgFwd(const R& res, double b, bool f, bool rf)
      : Row<R, MEM>(res), beta(b), first(f), refresh(rf) {}
  __device__ __forceinline__ void pre(int slot, int e) {
    this->begin(slot, e);
    h = this->get(refresh ? kR : kH);
    z = p = q = g = ds = 0.0;
    if (!refresh) {
      if (this->k.o.dsig) ds = this->k.o.dsig[3 * (int64_t)slot + e];
      z = ld<MEM>(this->zw(this->k.par, slot) + e);
      if (!first) {
        p = this->get(kP);
        q = this->get(kQ);
        g = this->get(kG);
      }
    }
  }
  __device__ __forceinline__ void post(int slot, int e, bool writes, const double (&s)[2]) {
    const double az = s[0] + h + ds * z;
    const double t = (refresh ? h : az) - s[1];
    const double w = this->solve(t, e);
    if (!writes) return;
    this->put_zw(this->zw(refresh ? this->k.next_copy() : this->k.par, slot) + 3 + e, unmarked(w));
    if (refresh) {
      this->put(kH, t);
    } else {
      p = z + beta * p;
      q = az + beta * q;
      g = t + beta * g;
      this->put(kP, p);
      this->put(kQ, q);
      this->put(kG, g);
      acc[0] += p * q;
    }
  }
};

// ---- phases outside the sweeps -------------------------------------------------
// x += alpha p, and r -= alpha q with the partial r.r unless the iteration
// recomputes the residual
template <int T, int K, int MEM>
__device__ __forceinline__ double cg_update_phase(const Resident<T, K, MEM>& k, double alpha, bool with_r) {
  const ResidentOp& o = k.o;
  double acc = 0.0;
#pragma unroll 1
  for (int64_t i = (int64_t)k.blk * T + threadIdx.x; i < 3 * (int64_t)o.ns; i += (int64_t)k.G * T) {
    double* b = rec(o, (int)(i / 3)) + (i % 3) * kRowsS;
    st<MEM>(b + kX * kRowsS, ld<MEM>(b + kX * kRowsS) + alpha * ld<MEM>(b + kP * kRowsS));
    if (with_r) {
      const double v = ld<MEM>(b + kR * kRowsS) - alpha * ld<MEM>(b + kQ * kRowsS);
      st<MEM>(b + kR * kRowsS, v);
      acc += v * v;
    }
  }
  drain_stores();
  return acc;
}
// x into the caller's node order
template <int T, int K, int MEM>
__device__ __forceinline__ void x_to_nodes(const Resident<T, K, MEM>& k) {
  const ResidentOp& o = k.o;
#pragma unroll 1
  for (int64_t i = (int64_t)k.blk * T + threadIdx.x; i < o.n; i += (int64_t)k.G * T) {
    const double* b = rec(o, o.node_slot[i]) + kX * kRowsS;
#pragma unroll
    for (int e = 0; e < 3; ++e) o.xn[3 * i + e] = ld<MEM>(b + e * kRowsS);
  }
}
// r = b - A x over the natural rows (x in o.xn), partial r.r
template <int T, int K, int MEM>
__device__ __forceinline__ double true_resid_phase(const Resident<T, K, MEM>& k) {
#pragma clang fp contract(off)
  const ResidentOp& o = k.o;
  double acc = 0.0;
#pragma unroll 1
  for (int s = k.blk * (T / kWave) + k.wave; s < o.A.nslices; s += k.G * (T / kWave)) {
    double y[3], xo[3];
    sell_row<2>(o.A, s, k.lane, o.xn, y, xo);
    const int64_t row = (int64_t)s * kRowsA + k.lane;
    if (row < o.n) {
      double* b = rec(o, o.node_slot[row]) + kR * kRowsS;
#pragma unroll
      for (int e = 0; e < 3; ++e) {
        const double v = o.b[3 * row + e] - y[e];
        st<MEM>(b + e * kRowsS, v);
        acc += v * v;
      }
    }
  }
  drain_stores();
  return acc;
}

// `budget` CG iterations (hecmw_solver_CG.f90:164-279) from the state in o.state;
// bit 0 of its `resume` says that z and rho stand as an earlier launch left them
// (else r and x do), bit 1 is the present copy.  Every thread runs the scalar logic on
// the same totals.
template <int T, int K, int MEM>
__global__ __launch_bounds__(T) void k_resident_cg(ResidentOp o, int budget) {
  extern __shared__ double lds[];
  using Res = Resident<T, K, MEM>;
  Res k(o, lds);
  KrylovState& st = *o.state;
  double rho = st.rho, rho1 = st.rho1, alpha = st.alpha, resid = st.resid, dnrm2 = st.dnrm2, c1 = st.c1;
  const double bnrm2 = st.bnrm2, tol = st.tol;
  int iter = st.iter, n_indef = st.n_indef, error = 0;
  const int maxit = st.maxit, nrec = st.nrec;
  const bool writer = blockIdx.x == 0 && threadIdx.x == 0;
  bool refresh = !(st.resume & 1);  // h and z have to be made from r first
  bool done = false, xn_current = false;
  uint64_t ticks[2] = {0, 0};  // forward and backward sweeps
  k.par = st.resume >> 1;
  k.begin(0);

#pragma unroll 1
  for (int n = 0; n < budget; ++n) {
    bool ended = false;  // the iteration's x and r stand without a backward sweep
    const bool upd = !refresh, periodic = iter % nrec == 0;
    uint64_t t0 = wall_clock64();
    {
      RowCgFwd<Res, MEM> f(k, iter > 1 ? rho / rho1 : 0.0, iter == 1, refresh);
      if (refresh) k.enter(k.next_copy());
      k.template sweep<2>(0, refresh ? k.next_copy() : k.par, f, !refresh);
      double tot[1];
      k.reduce(f.acc, tot);
      if (!refresh) c1 = tot[0];
    }
    uint64_t t1 = wall_clock64();
    ticks[refresh ? 1 : 0] += t1 - t0;
    if (!refresh) {
      if (c1 <= 0.0) {
        error = kErrDivergeMat;
        done = true;
      } else if (c1 != c1) {
        error = kErrDivergeNan;
        done = true;
      }
      if (done) break;
      alpha = rho / c1;
      xn_current = false;
      if (periodic || iter >= maxit) {
        double v[1] = {cg_update_phase(k, alpha, !periodic)}, tot[1];
        k.reduce(v, tot);
        if (!periodic) dnrm2 = tot[0];
        ended = true;
      }
    }
    double rho_next = 0.0;
    if (!ended) {
      k.par = k.next_copy();
      k.enter(k.par);
      RowCgBack<Res, MEM> f(k, alpha, upd);
      k.template sweep<1>(1, k.par, f);
      double tot[2];
      k.reduce(f.acc, tot);
      if (!upd) k.drop_lines();  // the refresh wrote, and this sweep marked, the same copy's w
      if (upd) dnrm2 = tot[0];
      rho_next = tot[1];
      ticks[1] += wall_clock64() - t1;
    }
    if (upd) {
      // the end of an iteration: convergence on a recomputed residual only
      if (!(ended && periodic)) {
        resid = sqrt(dnrm2 / bnrm2);
        if (writer) o.hist[iter - 1] = resid;
      }
      if ((ended && periodic) || resid <= tol) {
        x_to_nodes(k);
        k.full_sync();
        double v[1] = {true_resid_phase(k)}, tot[1];
        k.reduce(v, tot);
        dnrm2 = tot[0];
        resid = sqrt(dnrm2 / bnrm2);
        xn_current = true;
        if (writer && periodic) o.hist[iter - 1] = resid;
        done = resid <= tol;
        ended = true;
      }
      if (done) break;
      if (iter >= maxit) {
        error = kErrNoconv;
        iter = maxit + 1;
        done = true;
        break;
      }
      rho1 = rho;
      ++iter;
      if (ended) {
        refresh = true;
        k.begin(0);
        continue;
      }
    }
    rho = rho_next;
    refresh = false;
    if (rho == 0.0) {
      done = true;
    } else if (iter > 1 && rho * rho1 <= 0.0) {
      n_indef += 1;
      if (n_indef >= 3) {
        error = kErrDivergePc;
        done = true;
      }
    } else if (rho != rho) {
      error = kErrDivergeNan;
      done = true;
    }
    if (done) break;
  }
  if (!xn_current) x_to_nodes(k);
  if (writer) {
    st.rho = rho;
    st.rho1 = rho1;
    st.alpha = alpha;
    st.resid = resid;
    st.dnrm2 = dnrm2;
    st.c1 = c1;
    st.iter = iter;
    st.n_indef = n_indef;
    st.error = error;
    st.done = done ? 1 : 0;
    st.resume = (refresh ? 0 : 1) | k.par << 1;
    st.time_Ax += 1e-8 * (double)ticks[0];
    st.time_precond += 1e-8 * (double)ticks[1];
  }
  if (MEM == kOneGroup) {
    __syncthreads();
    for (int64_t i = threadIdx.x; i < o.ring * k.copy_size; i += T) o.zw[i] = k.zw0[i];
  }
}

// ---- BiCGSTAB (hecmw_solver_BiCGSTAB.f90:164-275) ---------------------------------
// The same two sweeps give p^ = M^-1 p, v = A p^ and s^ = M^-1 s, t = A s^; all
// other vectors are linear combinations, so their D'-multiplied transforms h =
// D' (D'+L)^-1 (.) follow by the same combinations (hr, hp of r and p, hv, ht from
// the forward sweeps of v and t).  s and hs replace r and hr (the reference too
// keeps s in r's place).

// backward row of p^ (half 0) or s^ (half 1)
template <class R, int MEM>
struct RowBiBack : Row<R, MEM> {
  int half;
  bool first, mark_w;
  double alpha, beta, omega;
  double r, hr, v, hv, p, hp, x, pt;
  __device__ __forceinline__ RowBiBack(const R& res, int hf, bool f, bool mw, double al, double be, double om)
      : Row<R, MEM>(res), half(hf), first(f), mark_w(mw), alpha(al), beta(be), omega(om) {}
  __device__ __forceinline__ void pre(int slot, int e) {
    this->begin(slot, e);
    r = this->get(kR);
    hr = this->get(kHr);
    if (half || !first) {
      v = this->get(kV);
      hv = this->get(kHv);
    }
    if (half) {
      x = this->get(kX);
      pt = ld<MEM>(this->zw(this->k.last_copy(), slot) + e);
    } else if (!first) {
      p = this->get(kBp);
      hp = this->get(kHp);
    }
  }
  __device__ __forceinline__ void post(int slot, int e, bool writes, const double (&s)[1]) {
    if (half) {
      r = r - alpha * v;
      hr = hr - alpha * hv;
      x = x + alpha * pt;
    } else {
      p = first ? r : r + beta * (p - omega * v);
      hp = first ? hr : hr + beta * (hp - omega * hv);
    }
    const double z = this->solve((half ? hr : hp) - s[0], e);
    if (!writes) return;
    double* now = this->zw(this->k.par, slot) + e;
    double* old = this->zw(this->k.last_copy(), slot) + e;
    this->put_zw(now, unmarked(z));
    this->put_zw(old, mark());
    this->put_zw(old + 3, mark());
    if (mark_w) this->put_zw(now + 3, mark());
    if (half) {
      this->put(kR, r);
      this->put(kHr, hr);
      this->put(kX, x);
    } else {
      this->put(kBp, p);
      this->put(kHp, hp);
    }
  }
};

// forward row of v (half 0) or t (half 1); refresh: only hr from r
template <class R, int MEM>
struct RowBiFwd : Row<R, MEM> {
  int half;
  bool refresh;
  double acc[2] = {0.0, 0.0};  // r~.v; t.s, t.t
  double h, z, u, ds;
  __device__ __forceinline__ RowBiFwd(const R& res, int hf, bool rf) : Row<R, MEM>(res), half(hf), refresh(rf) {}
  __device__ __forceinline__ void pre(int slot, int e) {
    this->begin(slot, e);
    h = this->get(refresh ? kR : (half ? kHr : kHp));
    z = u = ds = 0.0;
    if (!refresh) {
      if (this->k.o.dsig) ds = this->k.o.dsig[3 * (int64_t)slot + e];
      z = ld<MEM>(this->zw(this->k.par, slot) + e);
      u = this->get(half ? kR : kRt);
    }
  }
  __device__ __forceinline__ void post(int slot, int e, bool writes, const double (&s)[2]) {
    const double az = s[0] + h + ds * z;
    const double t = (refresh ? h : az) - s[1];
    const double w = this->solve(t, e);
    if (!writes) return;
    this->put_zw(this->zw(refresh ? this->k.next_copy() : this->k.par, slot) + 3 + e, unmarked(w));
    if (refresh) {
      this->put(kHr, t);
    } else {
      this->put(half ? kT : kV, az);
      this->put(half ? kHt : kHv, t);
      acc[0] += u * az;
      acc[1] += az * az;
    }
  }
};

// x += omega s^, and r = s - omega t, hr = hs - omega ht with the partials r.r and
// r~.r unless the iteration recomputes the residual
template <class R, int MEM>
__device__ __forceinline__ void bi_update_phase(const R& k, double omega, bool with_r, double (&acc)[2], int T) {
  const ResidentOp& o = k.o;
#pragma unroll 1
  for (int64_t i = (int64_t)k.blk * T + threadIdx.x; i < 3 * (int64_t)o.ns; i += (int64_t)k.G * T) {
    const int slot = (int)(i / 3), e = (int)(i % 3);
    if (o.row_old[slot] < 0) continue;
    double* b = rec(o, slot) + e * kRowsS;
    st<MEM>(b + kX * kRowsS, ld<MEM>(b + kX * kRowsS) + omega * ld<MEM>(k.zw(k.par, slot) + e));
    if (with_r) {
      const double v = ld<MEM>(b + kR * kRowsS) - omega * ld<MEM>(b + kT * kRowsS);
      st<MEM>(b + kR * kRowsS, v);
      st<MEM>(b + kHr * kRowsS, ld<MEM>(b + kHr * kRowsS) - omega * ld<MEM>(b + kHt * kRowsS));
      acc[0] += v * v;
      acc[1] += v * ld<MEM>(b + kRt * kRowsS);
    }
  }
  drain_stores();
}
// r~.r of a recomputed residual
template <class R, int MEM>
__device__ __forceinline__ double bi_rho_phase(const R& k, int T) {
  const ResidentOp& o = k.o;
  double acc = 0.0;
#pragma unroll 1
  for (int64_t i = (int64_t)k.blk * T + threadIdx.x; i < 3 * (int64_t)o.ns; i += (int64_t)k.G * T) {
    const double* b = rec(o, (int)(i / 3)) + i % 3 * kRowsS;
    acc += ld<MEM>(b + kR * kRowsS) * ld<MEM>(b + kRt * kRowsS);
  }
  return acc;
}

// `budget` BiCGSTAB iterations, as k_resident_cg
template <int T, int K, int MEM>
__global__ __launch_bounds__(T) void k_resident_bicg(ResidentOp o, int budget) {
  extern __shared__ double lds[];
  using Res = Resident<T, K, MEM>;
  Res k(o, lds);
  KrylovState& st = *o.state;
  double rho = st.rho, rho1 = st.rho1, alpha = st.alpha, omega = st.omega, resid = st.resid, dnrm2 = st.dnrm2;
  double c2 = st.c2, ts = st.ts, tt = st.tt;
  const double bnrm2 = st.bnrm2, tol = st.tol;
  int iter = st.iter, error = 0;
  const int maxit = st.maxit, nrec = st.nrec;
  const bool writer = blockIdx.x == 0 && threadIdx.x == 0;
  bool refresh = !(st.resume & 1);  // hr has to be made from r first
  bool done = false, xn_current = false;
  uint64_t ticks[2] = {0, 0};  // forward and backward sweeps
  k.par = st.resume >> 1;
  int half = 0;
  bool after_refresh = false;
  k.begin(refresh ? 0 : 1);

#pragma unroll 1
  for (int n = 0; n < budget;) {
    // p^ or s^, unless hr is made first
    if (!refresh) {
      const uint64_t t0 = wall_clock64();
      k.par = k.next_copy();
      k.enter(k.par);
      const double beta = iter > 1 ? (rho / rho1) * (alpha / omega) : 0.0;
      RowBiBack<Res, MEM> f(k, half, iter == 1, after_refresh, alpha, beta, omega);
      k.template sweep<1>(1, k.par, f);
      k.grid_sync();
      if (after_refresh) k.drop_lines();  // the refresh wrote, and this sweep marked, the same copy's w
      after_refresh = false;
      ticks[1] += wall_clock64() - t0;
    }
    double tot[2];
    {
      const uint64_t t0 = wall_clock64();
      RowBiFwd<Res, MEM> f(k, half, refresh);
      if (refresh) k.enter(k.next_copy());
      k.template sweep<2>(0, refresh ? k.next_copy() : k.par, f, !refresh);
      k.reduce(f.acc, tot);
      ticks[refresh ? 1 : 0] += wall_clock64() - t0;
    }
    if (refresh) {
      double v[1] = {bi_rho_phase<Res, MEM>(k, T)}, t[1];
      k.reduce(v, t);
      rho = t[0];
      refresh = false;
      after_refresh = true;
      continue;
    }
    if (half == 0) {
      c2 = tot[0];
      alpha = rho / c2;
      half = 1;
      continue;
    }
    half = 0;
    ts = tot[0];
    tt = tot[1];
    omega = ts / tt;
    const bool periodic = iter % nrec == 0;
    {
      double v[2] = {0.0, 0.0};
      bi_update_phase<Res, MEM>(k, omega, !periodic, v, T);
      k.reduce(v, tot);
    }
    xn_current = false;
    if (!periodic) {
      dnrm2 = tot[0];
      resid = sqrt(dnrm2 / bnrm2);
      if (writer) o.hist[iter - 1] = resid;
    }
    bool again = false;
    if (periodic || resid <= tol) {
      x_to_nodes(k);
      k.full_sync();
      double v[1] = {true_resid_phase(k)}, t[1];
      k.reduce(v, t);
      dnrm2 = t[0];
      resid = sqrt(dnrm2 / bnrm2);
      xn_current = true;
      if (writer && periodic) o.hist[iter - 1] = resid;
      done = resid <= tol;
      again = true;
    }
    if (done) break;
    if (iter >= maxit) {
      error = kErrNoconv;
      iter = maxit + 1;
      done = true;
      break;
    }
    rho1 = rho;
    rho = tot[1];
    ++iter;
    ++n;
    if (again) {
      refresh = true;
      k.begin(0);
    }
  }
  if (!xn_current) x_to_nodes(k);
  if (writer) {
    st.rho = rho;
    st.rho1 = rho1;
    st.alpha = alpha;
    st.omega = omega;
    st.c2 = c2;
    st.ts = ts;
    st.tt = tt;
    st.resid = resid;
    st.dnrm2 = dnrm2;
    st.iter = iter;
    st.error = error;
    st.done = done ? 1 : 0;
    st.resume = (refresh ? 0 : 1) | k.par << 1;
    st.time_Ax += 1e-8 * (double)ticks[0];
    st.time_precond += 1e-8 * (double)ticks[1];
  }
  if (MEM == kOneGroup) {
    __syncthreads();
    for (int64_t i = threadIdx.x; i < o.ring * k.copy_size; i += T) o.zw[i] = k.zw0[i];
  }
}

// ---- set-up ------------------------------------------------------------------
// the blocks of every row from its SELL slice into the lanes of its task: K
// consecutive blocks to a lane
__global__ __launch_bounds__(kBlock) void k_pack(Sell<double> s, const int2* __restrict__ row, int packets,
                                                   int32_t* __restrict__ col, double* __restrict__ val, int with_col) {
  const int64_t n = (int64_t)s.nslices * s.rows;
  // a quad per row, so that consecutive lanes write consecutive slots
  for (int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x; i < 4 * n; i += (int64_t)gridDim.x * kBlock) {
    const int64_t slot = i >> 2;
    const int64_t sl = slot / s.rows, r = slot - sl * s.rows, base = s.ptr[sl];
    const int len = s.len[slot];
    for (int k = (int)(i & 3); k < len; k += 4) {
      const int64_t at = (int64_t)row[slot].x + k / packets, g = at / kWave * packets + k % packets, l = at % kWave;
#pragma unroll
      for (int e = 0; e < 9; ++e) val[aval_index(g, e, (int)l)] = s.val[((base + k) * 9 + e) * s.rows + r];
      if (with_col) col[g * kWave + l] = s.col[(base + k) * s.rows + r];
    }
  }
}

// (1 - sigma) diag(D) of every row slot
__global__ __launch_bounds__(kBlock) void k_dsig(int32_t ns, const int32_t* __restrict__ row_old,
                                                   const double* __restrict__ D, double sigma, double* __restrict__ out) {
  for (int64_t t = (int64_t)blockIdx.x * kBlock + threadIdx.x; t < ns; t += (int64_t)gridDim.x * kBlock) {
    const int32_t i = row_old[t];
#pragma unroll
    for (int e = 0; e < 3; ++e) out[3 * t + e] = i >= 0 ? (1.0 - sigma) * D[9 * (int64_t)i + 4 * e] : 0.0;
  }
}

// the LU factors into the row records
__global__ __launch_bounds__(kBlock) void k_rec_alu(ResidentOp o, const double* __restrict__ alu, int rows) {
  for (int64_t t = (int64_t)blockIdx.x * kBlock + threadIdx.x; t < o.ns; t += (int64_t)gridDim.x * kBlock) {
    const double* f = alu + t / rows * 9 * rows + t % rows;
    double* b = rec(o, (int)t) + kAlu * kRowsS;
#pragma unroll
    for (int e = 0; e < 9; ++e) b[e * kRowsS] = f[e * rows];
  }
}

// r and x into slot order, the other vectors to zero, the gathered ones marked
__global__ __launch_bounds__(kBlock) void k_resident_init(ResidentOp o, const double* __restrict__ r, int zw_rec) {
  const int64_t i0 = (int64_t)blockIdx.x * kBlock + threadIdx.x, stride = (int64_t)gridDim.x * kBlock;
  // all entries marked, except the last record, which the unused blocks gather
  const int64_t nz = ((int64_t)o.ns + 1) * zw_rec;
  for (int64_t t = i0; t < o.ring * nz; t += stride) o.zw[t] = t % nz < (int64_t)o.ns * zw_rec ? mark() : 0.0;
  for (int64_t t = i0; t < o.ns; t += stride) {
    const int32_t i = o.row_old[t];
    double* b = rec(o, (int)t);
    for (int v = kR; v < o.planes; ++v) b[v * kRowsS] = 0.0;
#pragma unroll
    for (int e = 0; e < 3; ++e) {
      b[(kR + e) * kRowsS] = i >= 0 ? r[3 * (int64_t)i + e] : 0.0;
      b[(kX + e) * kRowsS] = i >= 0 ? o.xn[3 * (int64_t)i + e] : 0.0;
      if (o.planes == kBiPlanes) b[(kRt + e) * kRowsS] = b[(kR + e) * kRowsS];  // r~ = r0
    }
  }
}

// every launch starts with the exchange's entries marked
__global__ void k_resident_reset(uint32_t* sync) { reset_sync(sync); }

template <int T, int K, int MEM>
hipError_t launch(const ResidentOp& o, int grid, int budget, hipStream_t s) {
  const auto f = o.planes == kBiPlanes ? k_resident_bicg<T, K, MEM> : k_resident_cg<T, K, MEM>;
  const size_t lds = LdsMap<T>::bytes(o.ncolor, MEM == kOneGroup ? o.ns : 0);
  if (hipError_t e = allow_lds(reinterpret_cast<const void*>(f))) return e;
  k_resident_reset<<<1, 256, 0, s>>>(o.sync);
  ResidentOp op = o;
  void* args[] = {&op, &budget};
  return hipLaunchCooperativeKernel(reinterpret_cast<const void*>(f), dim3(grid), dim3(T), args, lds, s);
}

}  // namespace

void resident_pack(const Sell<double>& s, const int2* row, int packets, int32_t* col, double* val, bool with_col,
                   hipStream_t st) {
  const int64_t n = 4 * (int64_t)s.nslices * s.rows;
  k_pack<<<(int)std::min<int64_t>((n + kBlock - 1) / kBlock, 8192), kBlock, 0, st>>>(s, row, packets, col, val,
                                                                                    with_col ? 1 : 0);
}
void resident_dsig(int32_t ns, const int32_t* row_old, const double* D, double sigma, double* out, hipStream_t st) {
  k_dsig<<<std::min((ns + kBlock - 1) / kBlock, 2048), kBlock, 0, st>>>(ns, row_old, D, sigma, out);
}
void resident_alu(const ResidentOp& o, const double* alu, int rows, hipStream_t st) {
  k_rec_alu<<<std::min(std::max((o.ns + kBlock - 1) / kBlock, 1), 2048), kBlock, 0, st>>>(o, alu, rows);
}
void resident_init(const ResidentOp& o, const ResidentShape& sh, const double* r, hipStream_t st) {
  k_resident_init<<<std::min(std::max((o.ns + kBlock - 1) / kBlock, 1), 2048), kBlock, 0, st>>>(o, r, sh.grid == 1 ? 6 : 8);
}
bool resident_one_group(int ncolor, int ns) { return LdsMap<512>::bytes(ncolor, ns) <= kLdsBytes; }

hipError_t resident_run(const ResidentOp& o, const ResidentShape& sh, int budget, hipStream_t s) {
  if (sh.grid == 1) {
    switch (sh.packets) {
      case 2: return launch<512, 2, kOneGroup>(o, 1, budget, s);
      default: return launch<512, 4, kOneGroup>(o, 1, budget, s);
    }
  }
  switch (sh.packets) {
    case 2: return launch<512, 2, kGrid>(o, sh.grid, budget, s);
    default: return launch<512, 4, kGrid>(o, sh.grid, budget, s);
  }
}

}  // namespace hecmw33
