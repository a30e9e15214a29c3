// Linear solve of the assembled tangent on the device: Jacobi-preconditioned BiCGStab over
// the handle's CSR pattern (the system the reference hands to hypre GMRES + Euclid,
// src/solvers/hypre/Hypre.cc, once per global Newton iteration).
//
// One iteration is five launches and no host work: the scalars (rho, alpha, omega, the residual
// norm) stay on the device.  A kernel that closes a dot product leaves one partial per block;
// the next kernel's blocks each sum those partials in the same order, so every block has the
// same scalar, bit for bit, without an atomic, a second launch or a copy to the host.
//   step_p    res and rho from the last update; stop, or p <- r + beta (p - omega v), ph = D p
//   spmv V    v = A ph                        partials rh.v
//   step_s    alpha; r <- s = r - alpha v, sh = D s
//   spmv T    t = A sh                        partials t.t, t.s
//   step_x    omega; x += alpha ph + omega sh, r <- s - omega t   partials rh.r, r.r
// A launch reads no scalar that it writes.  The stop is kept as the number of the launch that decided
// it, and only later launches return for it: the deciding launch's blocks, which may see the word
// written or not, all reach the decision by themselves.
// The host enqueues a few iterations at a time and looks, one batch behind, at a status word in
// pinned memory; once the stop is decided, the launches already enqueued return at their first
// load.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdint>

#include "pgf_device.h"

namespace pgf {
namespace {

// The sums keep one fixed order, whatever the launch shape: a dot product of n entries has
// dot_blocks(n) partials; partial b is the tree sum over t < 256 of the entries
// b * 256 + t + k * 256 * dot_blocks(n), k = 0, 1, ..., each a chain of fmas.  A row's product is
// sixteen chains of fmas over the columns lane, lane + 16, ..., summed as a tree.
constexpr int kBlock = 256;
constexpr int kSpmvBlock = 512;
constexpr int kCols = 3;         // columns of a row group in flight per lane
constexpr int kMaxPart = 1024;   // partials of one dot product
constexpr int kBatch = 4;        // iterations between two looks at the status
constexpr int kLanes = 16;       // lanes of one row group: a DPP row, so its sums need no LDS

inline int dot_blocks(int64_t n) { return int(std::min<int64_t>(kMaxPart, (n + kBlock - 1) / kBlock)); }

struct Scalars {
  double rho[2], alpha, omega, bnorm, res;
  int64_t stop;  // the launch that decided the stop, kRunning before
  int32_t stop_after;
};
constexpr int64_t kRunning = INT64_MAX;
// launches are numbered over the solve, five an iteration in the order above
__host__ __device__ constexpr int64_t launch_number(int it, int k) { return 5 * int64_t(it) + k; }
// an earlier launch has decided the stop
__device__ __forceinline__ bool stopped(const Scalars *sc, int64_t launch) {
  return __hip_atomic_load(&sc->stop, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP) < launch;
}

template <int ROR>
__device__ __forceinline__ double row_rotate(double v) {  // lane i of a DPP row reads lane i - ROR mod 16
  const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(v), 0x120 + ROR, 0xf, 0xf, false);
  const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(v), 0x120 + ROR, 0xf, 0xf, false);
  return __hiloint2double(hi, lo);
}
// Tree sum over the 16 lanes of a DPP row (strides 8, 4, 2, 1): after each step the values
// repeat with the step's stride, so a rotation is the butterfly's exchange and every lane ends
// with the same bits.
__device__ __forceinline__ double row_sum(double v) {
  v += row_rotate<8>(v);
  v += row_rotate<4>(v);
  v += row_rotate<2>(v);
  v += row_rotate<1>(v);
  return v;
}
// Tree sums of the first 256 threads' a and b (strides 128, 64, ..., 1), on every thread.
__device__ __forceinline__ void tree_sum2(double &a, double &b) {
  __shared__ double sm[2][kBlock];
  __syncthreads();  // an earlier call's values have been read
  if (threadIdx.x < kBlock) {
    sm[0][threadIdx.x] = a;
    sm[1][threadIdx.x] = b;
  }
  __syncthreads();
  const int l = threadIdx.x & 63;
  a = (sm[0][l] + sm[0][l + 128]) + (sm[0][l + 64] + sm[0][l + 192]);
  b = (sm[1][l] + sm[1][l + 128]) + (sm[1][l + 64] + sm[1][l + 192]);
  a += __shfl_xor(a, 32);
  b += __shfl_xor(b, 32);
  a += __shfl_xor(a, 16);
  b += __shfl_xor(b, 16);
  a = row_sum(a);
  b = row_sum(b);
}
// The two dot products whose partials are pa[0..m) and pb[0..m).
__device__ __forceinline__ void close_dots(const double *pa, const double *pb, int m, double &a, double &b) {
  a = b = 0.0;
  if (threadIdx.x < kBlock)
    for (int i = threadIdx.x; i < m; i += kBlock) {
      a += pa[i];
      b += pb[i];
    }
  tree_sum2(a, b);
}

// What spmv does with A x besides storing it.
enum { kInit, kV, kT };

struct SpmvArgs {
  RowGroups rows;
  int64_t n;
  const int32_t *Ai;
  const double *vals, *x;
  double *y;                 // kV, kT: the product
  const double *w;           // kV: rh; kT: s; kInit: b
  double *r, *rh, *p, *v, *dinv;  // kInit
  double *pa, *pb;           // partials
  const Scalars *sc;
  int64_t launch;
};

__device__ __forceinline__ double pick3(int b, double v0, double v1, double v2) {
  return b == 0 ? v0 : (b == 1 ? v1 : v2);
}

// The rows of a node hold the same columns, so a group of 16 lanes takes the node's up to three
// rows together: a column index and the entry of x it picks are read once for three values.
// A workgroup takes the rows whose products its partial of the dot product sums (256-row
// ranges), so it forms the partial from what it has just stored.  Bound by the matrix's bytes
// (8 per entry + 4 per column of a node; 3.6 TB/s at 28.3 million entries, 74 us a product
// against 112 with a row to 16 lanes) and, below a range per CU, by the CU's rate of gathered
// entries of x (13 us at 1.46 million entries, 75 workgroups).
template <int MODE>
__global__ __launch_bounds__(kSpmvBlock) void spmv(SpmvArgs g) {
  if (MODE != kInit && stopped(g.sc, g.launch)) return;
  const int lane = threadIdx.x % kLanes;
  for (int rg = blockIdx.x; rg < g.rows.n_ranges; rg += gridDim.x) {
    const int hi = g.rows.range[rg + 1];
    for (int g0 = g.rows.range[rg]; g0 < hi; g0 += kSpmvBlock / kLanes) {
      const int gi = g0 + int(threadIdx.x) / kLanes;
      int4 row = make_int4(0, 0, 0, 0);
      if (gi < hi) row = g.rows.groups[gi];
      const int len = row.w;
      const double *v0 = g.vals + row.z, *v1 = v0 + (row.y > 1 ? len : 0), *v2 = v1 + (row.y > 2 ? len : 0);
      const int32_t *cols = g.Ai + row.z;
      double s0 = 0.0, s1 = 0.0, s2 = 0.0;
      double d0 = 0.0, d1 = 0.0, d2 = 0.0;  // kInit: the rows' diagonal entries, on the lanes that meet them
      for (int k0 = lane; k0 - lane < len; k0 += kCols * kLanes) {
        int c[kCols];
        double xv[kCols], a0[kCols], a1[kCols], a2[kCols];
#pragma unroll
        for (int j = 0; j < kCols; ++j) {  // past the row's end: its last entry, dropped below
          const int k = min(k0 + j * kLanes, len - 1);
          c[j] = cols[k];
          a0[j] = v0[k];
          a1[j] = v1[k];
          a2[j] = v2[k];
        }
#pragma unroll
        for (int j = 0; j < kCols; ++j) xv[j] = g.x[c[j]];
#pragma unroll
        for (int j = 0; j < kCols; ++j) {
          const bool in = k0 + j * kLanes < len;
          s0 = in ? __builtin_fma(a0[j], xv[j], s0) : s0;
          s1 = in ? __builtin_fma(a1[j], xv[j], s1) : s1;
          s2 = in ? __builtin_fma(a2[j], xv[j], s2) : s2;
          if constexpr (MODE == kInit) {
            d0 = in && c[j] == row.x ? a0[j] : d0;
            d1 = in && c[j] == row.x + 1 ? a1[j] : d1;
            d2 = in && c[j] == row.x + 2 ? a2[j] : d2;
          }
        }
      }
      s0 = row_sum(s0);
      s1 = row_sum(s1);
      s2 = row_sum(s2);
      if constexpr (MODE == kInit) {
        d0 = row_sum(d0);
        d1 = row_sum(d1);
        d2 = row_sum(d2);
      }
      if (lane < row.y) {
        const double ax = pick3(lane, s0, s1, s2);
        const int64_t i = int64_t(row.x) + lane;
        if constexpr (MODE == kInit) {
          const double r = g.w[i] - ax, d = pick3(lane, d0, d1, d2);
          g.dinv[i] = (d != 0.0 && isfinite(d)) ? 1.0 / d : 1.0;  // none, or not a number: 1
          g.r[i] = r;
          g.rh[i] = r;
          g.p[i] = 0.0;
          g.v[i] = 0.0;
        } else {
          g.y[i] = ax;
        }
      }
    }
  }
  __syncthreads();  // the workgroup's rows are stored
  double da = 0.0, db = 0.0;
  if (threadIdx.x < kBlock)
    for (int64_t i = int64_t(blockIdx.x) * kBlock + threadIdx.x; i < g.n; i += int64_t(gridDim.x) * kBlock) {
      const double w = g.w[i], y = MODE == kInit ? g.r[i] : g.y[i];
      if constexpr (MODE == kV) {
        da = __builtin_fma(w, y, da);
      } else if constexpr (MODE == kT) {
        da = __builtin_fma(y, y, da);
        db = __builtin_fma(y, w, db);
      } else {
        da = __builtin_fma(w, w, da);
        db = __builtin_fma(y, y, db);
      }
    }
  tree_sum2(da, db);
  if (threadIdx.x == 0) {
    g.pa[blockIdx.x] = da;
    if (MODE != kV) g.pb[blockIdx.x] = db;
  }
}

struct StepArgs {
  int64_t n;
  const double *dinv;
  double *r, *rh, *p, *v, *ph, *sh, *t, *x;
  const double *pa, *pb;  // partials this kernel closes
  int m;                  // their number
  double *qa, *qb;        // partials it leaves
  Scalars *sc;
  SolveStatus *status;    // pinned host memory
  double tol;
  int it, maxit;
  int64_t launch;
};

__device__ __forceinline__ void finish(const StepArgs &g, int it, double res) {
  __hip_atomic_store(&g.sc->stop, g.launch, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  g.status->it = it;
  g.status->res = res;
  __threadfence_system();
  g.status->done = 1;
}

// Iteration g.it: the state after iteration g.it - 1 decides whether it runs.
__global__ __launch_bounds__(kBlock) void step_p(StepArgs g) {
  if (stopped(g.sc, g.launch)) return;
  const bool first = g.it == 1, lead = blockIdx.x == 0 && threadIdx.x == 0;
  double a, b;
  close_dots(g.pa, g.pb, g.m, a, b);  // first: b.b and r.r (= rh.r); later: rh.r and r.r
  double bnorm, rho_old = 1.0, alpha = 1.0, omega = 1.0;
  if (first) {
    bnorm = sqrt(a);
    if (!(bnorm > 0.0)) bnorm = 1.0;
    a = b;
  } else {
    bnorm = g.sc->bnorm;
    rho_old = g.sc->rho[(g.it - 1) & 1];
    alpha = g.sc->alpha;
    omega = g.sc->omega;
  }
  const double res = sqrt(b) / bnorm;
  if (!(res > g.tol) || g.it > g.maxit || (!first && g.sc->stop_after)) {
    if (lead) finish(g, g.it - 1, res);
    return;
  }
  if (a == 0.0 || !isfinite(a)) {  // breakdown: the iteration counts, x stays
    if (lead) finish(g, g.it, res);
    return;
  }
  if (lead) {
    if (first) g.sc->bnorm = bnorm;
    g.sc->res = res;
    g.sc->rho[g.it & 1] = a;
  }
  const double beta = (a / rho_old) * (alpha / omega);
  for (int64_t i = int64_t(blockIdx.x) * kBlock + threadIdx.x; i < g.n; i += int64_t(gridDim.x) * kBlock) {
    const double p = __builtin_fma(beta, __builtin_fma(-omega, g.v[i], g.p[i]), g.r[i]);
    g.p[i] = p;
    g.ph[i] = g.dinv[i] * p;
  }
}

__global__ __launch_bounds__(kBlock) void step_s(StepArgs g) {
  if (stopped(g.sc, g.launch)) return;
  double rv, unused;
  close_dots(g.pa, g.pa, g.m, rv, unused);
  if (rv == 0.0 || !isfinite(rv)) {
    if (blockIdx.x == 0 && threadIdx.x == 0) finish(g, g.it, g.sc->res);
    return;
  }
  const double alpha = g.sc->rho[g.it & 1] / rv;
  if (blockIdx.x == 0 && threadIdx.x == 0) g.sc->alpha = alpha;
  for (int64_t i = int64_t(blockIdx.x) * kBlock + threadIdx.x; i < g.n; i += int64_t(gridDim.x) * kBlock) {
    const double s = __builtin_fma(-alpha, g.v[i], g.r[i]);
    g.r[i] = s;
    g.sh[i] = g.dinv[i] * s;
  }
}

__global__ __launch_bounds__(kBlock) void step_x(StepArgs g) {
  if (stopped(g.sc, g.launch)) return;
  double tt, ts;
  close_dots(g.pa, g.pb, g.m, tt, ts);
  const double omega = tt > 0.0 ? ts / tt : 0.0, alpha = g.sc->alpha;
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    g.sc->omega = omega;
    if (omega == 0.0) g.sc->stop_after = 1;
  }
  double da = 0.0, db = 0.0;
  for (int64_t i = int64_t(blockIdx.x) * kBlock + threadIdx.x; i < g.n; i += int64_t(gridDim.x) * kBlock) {
    g.x[i] = __builtin_fma(omega, g.sh[i], __builtin_fma(alpha, g.ph[i], g.x[i]));
    const double r = __builtin_fma(-omega, g.t[i], g.r[i]);
    g.r[i] = r;
    da = __builtin_fma(g.rh[i], r, da);
    db = __builtin_fma(r, r, db);
  }
  tree_sum2(da, db);
  if (threadIdx.x == 0) {
    g.qa[blockIdx.x] = da;
    g.qb[blockIdx.x] = db;
  }
}

__global__ void clear_scalars(Scalars *sc) {
  sc->stop = kRunning;
  sc->stop_after = 0;
}

}  // namespace

int64_t solve_work_doubles(int64_t n) {
  return 8 * n + 6 * kMaxPart + int64_t(sizeof(Scalars) / sizeof(double)) + 1;
}

int bicgstab(hipStream_t s, const RowGroups &rows, const int32_t *Ai, const double *vals, const double *b, double *x,
             int64_t n, double tol, int maxit, int *iters, double *relres, double *work, SolveStatus *status,
             hipEvent_t *ev) {
  if (n <= 0 || rows.n_ranges <= 0) return -1;
  double *r = work, *rh = r + n, *p = rh + n, *v = p + n, *ph = v + n, *sh = ph + n, *t = sh + n, *dinv = t + n,
         *part = dinv + n;
  auto *sc = reinterpret_cast<Scalars *>(part + 6 * kMaxPart);
  double *p_bb = part, *p_rr = part + kMaxPart, *p_rho = part + 2 * kMaxPart, *p_rv = part + 3 * kMaxPart,
         *p_tt = part + 4 * kMaxPart, *p_ts = part + 5 * kMaxPart;
  status->done = 0;
  status->it = 0;
  status->res = std::nan("");
  const unsigned nb = unsigned(dot_blocks(n));
  SpmvArgs m{rows, n, Ai, vals, x, nullptr, b, r, rh, p, v, dinv, p_bb, p_rr, sc, 0};
  StepArgs e{n, dinv, r, rh, p, v, ph, sh, t, x, p_bb, p_rr, int(nb), p_rho, p_rr, sc, status, tol, 0, maxit, 0};
  clear_scalars<<<1, 1, 0, s>>>(sc);
  spmv<kInit><<<nb, kSpmvBlock, 0, s>>>(m);
  hipError_t err = hipSuccess;
  auto chk = [&](hipError_t q) {
    if (q != hipSuccess && err == hipSuccess) err = q;
    return q == hipSuccess;
  };
  int it = 1;
  for (int batch = 0; err == hipSuccess; ++batch) {
    bool last = false;
    for (int k = 0; k < kBatch && !last; ++k, ++it) {
      e.it = it;
      e.launch = launch_number(it, 0);
      e.pa = it == 1 ? p_bb : p_rho;
      e.pb = p_rr;
      step_p<<<nb, kBlock, 0, s>>>(e);
      last = it > maxit;  // that launch only takes the last iteration's residual norm
      if (last) break;
      m.x = ph;
      m.y = v;
      m.w = rh;
      m.pa = p_rv;
      m.launch = launch_number(it, 1);
      spmv<kV><<<nb, kSpmvBlock, 0, s>>>(m);
      e.pa = p_rv;
      e.launch = launch_number(it, 2);
      step_s<<<nb, kBlock, 0, s>>>(e);
      m.x = sh;
      m.y = t;
      m.w = r;
      m.pa = p_tt;
      m.pb = p_ts;
      m.launch = launch_number(it, 3);
      spmv<kT><<<nb, kSpmvBlock, 0, s>>>(m);
      e.pa = p_tt;
      e.pb = p_ts;
      e.launch = launch_number(it, 4);
      step_x<<<nb, kBlock, 0, s>>>(e);
    }
    if (!chk(hipGetLastError()) || !chk(hipEventRecord(ev[batch & 1], s))) break;
    if (batch > 0 && (!chk(hipEventSynchronize(ev[(batch - 1) & 1])) || status->done)) break;
    if (last) break;
  }
  if (!chk(hipStreamSynchronize(s))) return -1;
  if (!status->done) return -1;
  *iters = status->it;
  *relres = status->res;
  return err == hipSuccess ? 0 : -1;
}

}  // namespace pgf
