// CG with block-diagonal scaling as one resident kernel that keeps its matrix in the
// register files.
//
// Launch by launch an iteration takes nine kernels, each with its gap and its trip of
// the vectors through memory, and reads all of A.  256 CUs hold 128 MB of registers
// and 40 MB of LDS: up to about 50,000 nodes the FP64 blocks of A fit the registers
// of one wave per SIMD and are read once per launch of many iterations, and all
// vectors but the gathered one stay in LDS.
//  * A task is up to 16 consecutive rows on 64 lanes, kDiagK blocks to a lane, a row
//    taking whole lanes: seven blocks fit the 27 of a HEX8 row into 4 lanes (28) and
//    the 18 of a face row into 3 (21).  A wave keeps its first R tasks in registers
//    and reads the others again every iteration.
//  * z = D^-1 r is the only gathered vector: w = A z, p = z + beta p and q = A p = w +
//    beta q, so that z is written before the reduction of r.z, whose grid barrier also
//    publishes it; the reduction of p.q is the only other barrier.
//  * The records of z rotate through a ring of copies: a copy's lines are in no cache
//    before they are read, so that plain loads through L1 and L2 serve the gathers
//    without an invalidation per iteration; one acquire fence per turn of the ring
//    clears the lines of the turn before.  A record is 32 bytes and a task's rows are
//    whole groups of four, so that no 128-byte line has two writers.
// Measured, us per iteration, launch by launch -> resident (HEX8 cubes): 729 nodes 32.8
// -> 6.3, 2,197 33 -> 7.0, 9,261 34 -> 8.7, 24,389 36 -> 10.8, 39,304 37 -> 14.8, 91,125
// 57 -> 38.  Up to one task per wave the two exchanges and the chain gather -> sums ->
// update bound it; with three, that chain three times over (one wave per SIMD has
// nothing beside it); beyond, the tasks that are read again (120 MB an iteration at
// 91,125 nodes).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>

#include "device.h"
#include "resident.h"
#include "rows.h"

namespace hecmw33 {
namespace {

constexpr int kThreads = 256;  // one wave per SIMD: 512 registers a lane
constexpr int kWavesD = kThreads / kWave;
// LDS of a task: the LU of its rows' D, and by lane x, r, p, q and z
constexpr int kTaskDoubles = 9 * kResidentRows + 5 * kWave;
constexpr int kScratchDoubles = kWavesD * 3 * kWave + GridGroup<kThreads, kGrid>::kRedDoubles;

struct Lane {
  int row, first;  // row in the task (-1: idle), first block
  __device__ __forceinline__ explicit Lane(int32_t m) : row(m < 0 ? -1 : m & 15), first((m >> 4 & 0x3ff) * kDiagK) {}
};

struct Blocks {
  double v[kDiagK][9];
  int32_t c[kDiagK];
};

// the lane's blocks of task t from the SELL-64 rows of A; blocks past the row's end
// are zero and gather the record that is always zero
__device__ __forceinline__ void load_blocks(const DiagOp& o, int t, int lane, Blocks& b) {
  const Lane m(o.lane[(int64_t)t * kWave + lane]);
  const int row = o.task[t].x + max(m.row, 0), r = row % kRowsA;
  const int len = m.row < 0 ? 0 : o.A.len[row];
  const int64_t base = (int64_t)o.A.ptr[row / kRowsA] + m.first;
#pragma unroll
  for (int k = 0; k < kDiagK; ++k) {
    b.c[k] = o.zero_rec;
#pragma unroll
    for (int e = 0; e < 9; ++e) b.v[k][e] = 0.0;
    if (m.first + k < len) {
      b.c[k] = o.A.col[(base + k) * kRowsA + r];
      aval_load(o.A.val, base + k, r, b.v[k]);
    }
  }
}

template <int R, bool STREAM, int MEM>
struct DiagCg : GridGroup<kThreads, MEM> {
  using Group = GridGroup<kThreads, MEM>;
  using Group::blk;
  using Group::G;
  using Group::lane;
  using Group::wave;
  const DiagOp& o;
  double *prod, *tasks;  // LDS: this wave's products, the workgroup's tasks
  int t0, nt;            // the workgroup's tasks
  int cp = -1;           // ring copy written last
  int sub, e;            // the lane's row in the row work, and its entry (the fourth mirrors the third)
  Blocks keep[R];
  Blocks next;           // STREAM: the next task to be read

  __device__ __forceinline__ DiagCg(const DiagOp& op, double* lds) : Group(op.sync, lds + kWavesD * 3 * kWave), o(op) {
    prod = lds + wave * 3 * kWave;
    tasks = lds + kScratchDoubles;
    t0 = (int)((int64_t)o.ntasks * blk / G);
    nt = (int)((int64_t)o.ntasks * (blk + 1) / G) - t0;
    sub = lane >> 2;
    e = (lane & 3) < 3 ? lane & 3 : 2;
#pragma unroll
    for (int q = 0; q < R; ++q)
      if (wave + q * kWavesD < nt) load_blocks(o, t0 + wave + q * kWavesD, lane, keep[q]);
    prefetch();
  }
  __device__ __forceinline__ void prefetch() {
    if (STREAM && wave + R * kWavesD < nt) load_blocks(o, t0 + wave + R * kWavesD, lane, next);
  }
  __device__ __forceinline__ double* lu(int i) const { return tasks + (int64_t)i * kTaskDoubles; }
  __device__ __forceinline__ double& vec(int i, int v) const { return lu(i)[9 * kResidentRows + v * kWave + lane]; }
  enum { X, R_, P, Q, Z };

  // f(task of the workgroup, rows, the lane's row) for every task of this wave
  template <class F>
  __device__ __forceinline__ void rows(F f) {
#pragma unroll 1
    for (int i = wave; i < nt; i += kWavesD) {
      const int4 d = o.task[t0 + i];
      f(i, d.y, d.x + sub);
    }
  }
  __device__ __forceinline__ void load_state(bool resumed) {
    rows([&](int i, int nr, int row) {
      const bool live = sub < nr && row < o.n;
      const int64_t at = 3 * (int64_t)row + e;
      vec(i, X) = live ? o.x[at] : 0.0;
      vec(i, R_) = live ? o.r[at] : 0.0;
      vec(i, P) = live && resumed ? o.p[at] : 0.0;
      vec(i, Q) = live && resumed ? o.q[at] : 0.0;
      if ((lane & 3) == 3) return;
      for (int k = 3 * e; k < 3 * e + 3; ++k)
        lu(i)[9 * sub + k] = live ? o.alu[((int64_t)(row / kRowsA) * 9 + k) * kRowsA + row % kRowsA] : 0.0;
    });
  }
  __device__ __forceinline__ void store_state() {
    rows([&](int i, int nr, int row) {
      if (sub >= nr || row >= o.n || (lane & 3) == 3) return;
      const int64_t at = 3 * (int64_t)row + e;
      o.x[at] = vec(i, X);
      o.r[at] = vec(i, R_);
      o.p[at] = vec(i, P);
      o.q[at] = vec(i, Q);
    });
  }

  __device__ __forceinline__ void next_copy() { cp = cp + 1 == o.ring ? 0 : cp + 1; }
  __device__ __forceinline__ void publish(int row, double y) {
    if ((lane & 3) < 3) st<MEM>(o.z + cp * o.copy + 4 * (int64_t)row + e, y);
  }
  // after the barrier that follows a publish: the lines of the ring's last turn go
  __device__ __forceinline__ void turn() {
    if (MEM == kGrid && cp == 0) __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
  }

  // the end of an iteration (upd) and z of the next: x += alpha p, r -= alpha q,
  // z = D^-1 r; acc: r.r, r.z
  __device__ __forceinline__ void update(bool upd, double alpha, double (&acc)[2]) {
    next_copy();
    rows([&](int i, int nr, int row) {
      double r = vec(i, R_);
      if (upd) {
        vec(i, X) += alpha * vec(i, P);
        r -= alpha * vec(i, Q);
        vec(i, R_) = r;
      }
      double a[9];
#pragma unroll
      for (int k = 0; k < 9; ++k) a[k] = lu(i)[9 * sub + k];
      double y0 = quad_bcast<0>(r), y1 = quad_bcast<1>(r), y2 = quad_bcast<2>(r);
      lu3_solve<double>(a, y0, y1, y2);
      const double z = e == 0 ? y0 : (e == 1 ? y1 : y2);
      if (sub < nr) {
        publish(row, z);
        vec(i, Z) = z;
        if ((lane & 3) < 3) {
          acc[0] += r * r;
          acc[1] += r * z;
        }
      }
    });
    drain_stores();
  }
  __device__ __forceinline__ void publish_x() {
    next_copy();
    rows([&](int i, int nr, int row) {
      if (sub < nr) publish(row, vec(i, X));
    });
    drain_stores();
  }

  template <class F>
  __device__ __forceinline__ void task(int i, const Blocks& b, F& f) {
    const double* z = o.z + cp * o.copy;
    double x[kDiagK][3];
#pragma unroll
    for (int k = 0; k < kDiagK; ++k) {
      const double* q = z + 4 * (int64_t)b.c[k];
      const double2 u = *reinterpret_cast<const double2*>(q);
      x[k][0] = u.x;
      x[k][1] = u.y;
      x[k][2] = q[2];
    }
    const int4 d = o.task[t0 + i];
    const int at = o.lane[(int64_t)(t0 + i) * kWave + lane] >> 14 & 63;
    const int2 info = o.row[d.x + min(sub, d.y - 1)];
#pragma unroll
    for (int j = 0; j < 3; ++j) {
      double s = 0.0;
#pragma unroll
      for (int k = 0; k < kDiagK; ++k)
        s = fma(b.v[k][3 * j + 2], x[k][2], fma(b.v[k][3 * j + 1], x[k][1], fma(b.v[k][3 * j], x[k][0], s)));
      prod[j * kWave + at] = s;
    }
    lds_order();
    if (sub < d.y) {
      const double* pr = prod + e * kWave + info.x;
      double sum = 0.0;
#pragma unroll 1
      for (int k = 0; k < info.y; k += 4) {
        double y[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) y[u] = pr[min(k + u, info.y - 1)];
#pragma unroll
        for (int u = 0; u < 4; ++u) sum += k + u < info.y ? y[u] : 0.0;
      }
      f(i, d.x + sub, sum);
    }
    lds_order();
  }
  // f(task, row, entry e of the row of A times the published vector) for the rows of this wave
  template <class F>
  __device__ __forceinline__ void product(F f) {
#pragma unroll
    for (int q = 0; q < R; ++q)
      if (wave + q * kWavesD < nt) task(wave + q * kWavesD, keep[q], f);
    if (STREAM) {
#pragma unroll 1
      for (int i = wave + R * kWavesD; i < nt; i += kWavesD) {
        task(i, next, f);
        if (i + kWavesD < nt) load_blocks(o, t0 + i + kWavesD, lane, next);
      }
      prefetch();
    }
  }
};

// `budget` CG iterations (hecmw_solver_CG.f90:164-279) from the state in o.state.  Every
// thread runs the scalar logic on the same totals.
template <int R, bool STREAM, int MEM>
__global__ __launch_bounds__(kThreads, 1) void k_resident_diag_cg(DiagOp o, int budget) {
  extern __shared__ double lds[];
  using Cg = DiagCg<R, STREAM, MEM>;
  Cg k(o, lds);
  KrylovState& st = *o.state;
  double rho = st.rho, rho1 = st.rho1, alpha = st.alpha, resid = st.resid, dnrm2 = st.dnrm2, c1 = st.c1;
  const double bnrm2 = st.bnrm2, tol = st.tol;
  int iter = st.iter, n_indef = st.n_indef, error = 0;
  const int maxit = st.maxit, nrec = st.nrec;
  const bool writer = blockIdx.x == 0 && threadIdx.x == 0;
  bool upd = false, done = false;  // upd: an iteration's x and r are still to be made
  uint64_t ticks[2] = {0, 0};  // products, the rest
  k.load_state(iter > 1);
  __syncthreads();

#pragma unroll 1
  for (int n = 0; n <= budget; ++n) {
    // the last pass of a launch only ends its iteration
    uint64_t t0 = wall_clock64();
    double acc[2] = {0.0, 0.0}, tot[2];
    k.update(upd, alpha, acc);
    k.reduce(acc, tot);
    k.turn();
    if (upd) {
      dnrm2 = tot[0];
      const bool periodic = iter % nrec == 0;
      if (!periodic) {
        resid = sqrt(dnrm2 / bnrm2);
        if (writer) o.hist[iter - 1] = resid;
      }
      bool again = false;
      if (periodic || resid <= tol) {
        // convergence on a recomputed residual only
        k.publish_x();
        k.grid_sync();
        k.turn();
        double v[1] = {0.0}, rr[1];
        k.product([&](int i, int row, double s) {
          const double r = row < o.n ? o.b[3 * (int64_t)row + k.e] - s : 0.0;
          k.vec(i, Cg::R_) = r;
          if ((k.lane & 3) < 3) v[0] += r * r;
        });
        k.reduce(v, rr);
        dnrm2 = rr[0];
        resid = sqrt(dnrm2 / bnrm2);
        if (writer && periodic) o.hist[iter - 1] = resid;
        done = resid <= tol;
        again = true;
      }
      upd = false;
      if (done) break;
      if (iter >= maxit) {
        error = kErrNoconv;
        iter = maxit + 1;
        done = true;
        break;
      }
      rho1 = rho;
      ++iter;
      if (again) {
        double a2[2] = {0.0, 0.0};
        k.update(false, 0.0, a2);
        k.reduce(a2, tot);
        k.turn();
      }
    }
    if (n == budget) break;
    rho = tot[1];
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
    const uint64_t t1 = wall_clock64();
    ticks[1] += t1 - t0;
    const double beta = iter > 1 ? rho / rho1 : 0.0;
    double pq[1] = {0.0};
    k.product([&](int i, int row, double s) {
      const double p = k.vec(i, Cg::Z) + beta * k.vec(i, Cg::P);
      const double q = s + beta * k.vec(i, Cg::Q);
      k.vec(i, Cg::P) = p;
      k.vec(i, Cg::Q) = q;
      if ((k.lane & 3) < 3) pq[0] += p * q;
    });
    double c[1];
    k.reduce(pq, c);
    c1 = c[0];
    ticks[0] += wall_clock64() - t1;
    if (c1 <= 0.0) {
      error = kErrDivergeMat;
      done = true;
    } else if (c1 != c1) {
      error = kErrDivergeNan;
      done = true;
    }
    if (done) break;
    alpha = rho / c1;
    upd = true;
  }
  k.store_state();
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
    st.time_Ax += 1e-8 * (double)ticks[0];
    st.time_precond += 1e-8 * (double)ticks[1];
  }
}

// the zero records of the ring's copies, and the entries of the exchange
__global__ void k_diag_reset(DiagOp o) {
  reset_sync(o.sync);
  for (int i = threadIdx.x; i < 4 * o.ring; i += blockDim.x)
    o.z[(i / 4) * o.copy + 4 * (int64_t)o.zero_rec + i % 4] = 0.0;
}

template <int R, bool STREAM, int MEM>
hipError_t launch(const DiagOp& o, int grid, int budget, hipStream_t s) {
  const auto f = k_resident_diag_cg<R, STREAM, MEM>;
  const size_t lds = diag_lds_bytes(o.ntasks, grid);
  if (hipError_t e = allow_lds(reinterpret_cast<const void*>(f))) return e;
  k_diag_reset<<<1, 256, 0, s>>>(o);
  DiagOp op = o;
  void* args[] = {&op, &budget};
  return hipLaunchCooperativeKernel(reinterpret_cast<const void*>(f), dim3(grid), dim3(kThreads), args, lds, s);
}
template <int MEM>
hipError_t launch_kept(const DiagOp& o, int grid, int budget, hipStream_t s) {
  const int per = ((o.ntasks + grid - 1) / grid + kWavesD - 1) / kWavesD;  // tasks of a wave
  if (per <= 1) return launch<1, false, MEM>(o, grid, budget, s);
  if (per <= 2) return launch<2, false, MEM>(o, grid, budget, s);
  if (per <= 3) return launch<3, false, MEM>(o, grid, budget, s);
  return launch<2, true, MEM>(o, grid, budget, s);
}

}  // namespace

size_t diag_lds_bytes(int ntasks, int grid) {
  return sizeof(double) * (kScratchDoubles + (size_t)((ntasks + grid - 1) / grid) * kTaskDoubles);
}

hipError_t resident_diag_run(const DiagOp& o, int grid, int budget, hipStream_t s) {
  return grid == 1 ? launch_kept<kOneGroup>(o, 1, budget, s) : launch_kept<kGrid>(o, grid, budget, s);
}

}  // namespace hecmw33
