// The LIS option strings beyond "-i cg -p jacobi": CG, CGS and BiCGSTAB with no,
// Jacobi or SSOR preconditioning, in FP64 on the device. The reference's default is
// "-p ssor -ssor_omega 0.51 -i cgs -tol 1.e-6" (src/pb_class.cpp:970,
// data/options.prm:174), handed to LIS through lis_solver_set_option
// (src/pb_class.cpp:2294-2315).
//
// Algorithms (LIS is not vendored with the reference; these are the published forms):
//   SSOR (Saad, Iterative Methods for Sparse Linear Systems, sec. 10.2): with
//   A = L + D + U, M = (D + w L) D^-1 (D + w U). M^-1 r is a forward sweep
//   y_i = (r_i - w sum_{j<i} a_ij y_j) / d_i, then a backward sweep
//   z_i = y_i - w (sum_{j>i} a_ij z_j) / d_i, each row's entries in ascending column
//   order with the arithmetic t = t - (w a_ij) y_j and t = t + a_ij z_j, so the result
//   is the oracle's bit for bit.
//   CGS and BiCGSTAB as in Barrett et al., Templates (1994), sec. 2.3.7-2.3.8, x0 = 0,
//   shadow residual r~ = b, stop when ||r||_2 <= tol ||b||_2 (BiCGSTAB also tests s).
//
// The sweeps are level-scheduled: a row's forward level is one more than the largest
// level among its lower neighbours (backward: upper neighbours), so the rows of one
// level are independent. The levels depend only on the sparsity pattern and are built
// once per pattern on the host from the CSR. Rows take positions in level order; a
// sweep's vectors and entries are packed in that order and name neighbours by position.
//
// A sweep is a serial chain of levels (427 on a 255,000-row protein mesh, 600 rows each
// on average), so its time is the chain's latency. Runs of narrow levels (order_triangle)
// go to one block (k_ssor_run), piece by piece (a piece: rows of one level that fit the
// staging buffers): the next pieces' entries stream into LDS while one is solved, the
// solution of the last kWindow positions stays in LDS, and pieces are separated by a
// block barrier. Wider levels, which fill more than one compute unit, are launched one by
// one (k_ssor_level).
//
// Reductions follow the FP64 CG: per-block partials, summed in a fixed order by a
// one-block finalize kernel that also updates the scalars and the stop flag; every
// kernel launched after the stop flag returns at once, and the host polls the flag
// every check_every iterations.
#include <algorithm>
#include <array>
#include <cmath>
#include <cstring>
#include <type_traits>
#include <vector>

#include "ngpb_internal.h"

namespace ngpb {
namespace {

constexpr int kBS = 256;
constexpr int kFin = 1024;

// KrylovScalars fields used here: rho, pq (denominator), alpha, beta, rr, stop_rr, bb,
// aux[0] omega, aux[1] rho of the previous iteration, aux[2] (s, s), aux[3] 1 once
// BiCGSTAB's s met the tolerance; iter, maxiter, done, status.
enum Fin : int { kFinRho = 0, kFinAlpha = 1, kFinResid = 2, kFinBicgS = 3, kFinOmega = 4, kFinBicgResid = 5,
                 kFinCgBeta = 6, kFinCgRho0 = 7 };

__global__ void __launch_bounds__(kBS) k_lis_init(int64_t n, const double* __restrict__ b, double* __restrict__ x,
                                                  double* __restrict__ r, double* __restrict__ rt,
                                                  double* __restrict__ p, double* __restrict__ q,
                                                  double* __restrict__ v, double* __restrict__ part) {
  __shared__ double s_red[kBS / 64];
  double bb = 0.0;
  for (int64_t i = (int64_t)blockIdx.x * kBS + threadIdx.x; i < n; i += (int64_t)gridDim.x * kBS) {
    const double bi = b[i];
    x[i] = 0.0;
    r[i] = bi;
    rt[i] = bi;
    p[i] = 0.0;
    q[i] = 0.0;
    v[i] = 0.0;
    bb += bi * bi;
  }
  bb = dev::block_sum<kBS>(bb, s_red);
  if (threadIdx.x == 0) part[2 * blockIdx.x] = bb;
}

__global__ void __launch_bounds__(kFin) k_lis_fin_init(KrylovScalars* ks, const double* __restrict__ part, int np,
                                                       double tol2, int maxiter) {
  __shared__ double s_red[kFin / 64];
  const double BB = dev::sum_partials<kFin>(part, np, 2, s_red);
  if (threadIdx.x == 0) {
    ks->bb = BB;
    ks->rr = BB;
    ks->stop_rr = tol2 * BB;
    ks->rho = 0.0;
    ks->pq = 0.0;
    ks->alpha = 1.0;
    ks->beta = 0.0;
    ks->aux[0] = 1.0;
    ks->aux[1] = 1.0;
    ks->aux[2] = 0.0;
    ks->aux[3] = 0.0;
    ks->iter = 0;
    ks->maxiter = maxiter;
    ks->status = 0;
    ks->done = (BB == 0.0) ? 1 : 0;
  }
}

// per-block partials of (a, b) and, with TWO, (c, d); stride 2
template <bool TWO>
__global__ void __launch_bounds__(kBS) k_dots(int64_t n, const double* __restrict__ a, const double* __restrict__ b,
                                              const double* __restrict__ c, const double* __restrict__ d,
                                              const KrylovScalars* ks, double* __restrict__ part) {
  __shared__ double s_red[kBS / 64];
  if (ks->done) return;
  double s1 = 0.0, s2 = 0.0;
  for (int64_t i = (int64_t)blockIdx.x * kBS + threadIdx.x; i < n; i += (int64_t)gridDim.x * kBS) {
    s1 += a[i] * b[i];
    if (TWO) s2 += c[i] * d[i];
  }
  s1 = dev::block_sum<kBS>(s1, s_red);
  if (TWO) s2 = dev::block_sum<kBS>(s2, s_red);
  if (threadIdx.x == 0) {
    part[2 * blockIdx.x] = s1;
    if (TWO) part[2 * blockIdx.x + 1] = s2;
  }
}

// One block: sums the partials in a fixed order and advances the scalar state.
__global__ void __launch_bounds__(kFin) k_lis_fin(KrylovScalars* ks, const double* __restrict__ part, int np,
                                                  int stride, int what, int solver) {
  __shared__ double s_red[kFin / 64];
  if (ks->done) return;
  const double S0 = dev::sum_partials<kFin>(part, np, stride, s_red);
  const double S1 = (what == kFinOmega) ? dev::sum_partials<kFin>(part + 1, np, stride, s_red) : 0.0;
  if (threadIdx.x != 0) return;
  const bool sconv = ks->aux[3] != 0.0;
  switch (what) {
    case kFinRho:  // rho = (r~, r) at the start of a CGS / BiCGSTAB iteration
      if (S0 == 0.0) {
        ks->done = 1;
        ks->status = NGPB_E_NOCONV;
        break;
      }
      ks->rho = S0;
      if (ks->iter == 0) ks->beta = 0.0;
      else if (solver == NGPB_SOLVER_CGS) ks->beta = S0 / ks->aux[1];
      else ks->beta = (S0 / ks->aux[1]) * (ks->alpha / ks->aux[0]);
      break;
    case kFinAlpha:  // alpha = rho / denominator
      ks->pq = S0;
      if (S0 == 0.0) {
        ks->done = 1;
        ks->status = NGPB_E_NOCONV;
        break;
      }
      ks->alpha = ks->rho / S0;
      break;
    case kFinResid:  // CG / CGS: stop test on the updated residual
      ks->rr = S0;
      ks->iter += 1;
      if (S0 <= ks->stop_rr) {
        ks->done = 1;
        ks->status = 0;
      } else if (ks->iter >= ks->maxiter) {
        ks->done = 1;
        ks->status = NGPB_E_NOCONV;
      } else {
        ks->aux[1] = ks->rho;
      }
      break;
    case kFinBicgS:  // BiCGSTAB: s = r - alpha v met the tolerance?
      ks->aux[2] = S0;
      ks->iter += 1;
      if (S0 <= ks->stop_rr) ks->aux[3] = 1.0;
      break;
    case kFinOmega:  // omega = (t, s) / (t, t)
      if (sconv) break;
      if (S0 == 0.0 || S1 == 0.0) {
        ks->done = 1;
        ks->status = NGPB_E_NOCONV;
        break;
      }
      ks->aux[0] = S0 / S1;
      break;
    case kFinBicgResid:
      if (sconv) {
        ks->rr = ks->aux[2];
        ks->done = 1;
        ks->status = 0;
        break;
      }
      ks->rr = S0;
      if (S0 <= ks->stop_rr) {
        ks->done = 1;
        ks->status = 0;
      } else if (ks->iter >= ks->maxiter) {
        ks->done = 1;
        ks->status = NGPB_E_NOCONV;
      } else {
        ks->aux[1] = ks->rho;
      }
      break;
    case kFinCgBeta: {  // CG: rho' = (r, z); beta = rho' / rho
      ks->beta = S0 / ks->rho;
      ks->rho = S0;
      break;
    }
    case kFinCgRho0:
      ks->rho = S0;
      break;
  }
}

// CGS: u = r + beta q; p = u + beta (q + beta p)
__global__ void __launch_bounds__(kBS) k_cgs_up(int64_t n, const double* __restrict__ r, const double* __restrict__ q,
                                                double* __restrict__ u, double* __restrict__ p, const KrylovScalars* ks) {
  if (ks->done) return;
  const double beta = ks->beta;
  for (int64_t i = (int64_t)blockIdx.x * kBS + threadIdx.x; i < n; i += (int64_t)gridDim.x * kBS) {
    const double ui = r[i] + beta * q[i];
    u[i] = ui;
    p[i] = ui + beta * (q[i] + beta * p[i]);
  }
}

// CGS: q = u - alpha v; t = u + q
__global__ void __launch_bounds__(kBS) k_cgs_q(int64_t n, const double* __restrict__ u, const double* __restrict__ v,
                                               double* __restrict__ q, double* __restrict__ t, const KrylovScalars* ks) {
  if (ks->done) return;
  const double alpha = ks->alpha;
  for (int64_t i = (int64_t)blockIdx.x * kBS + threadIdx.x; i < n; i += (int64_t)gridDim.x * kBS) {
    const double qi = u[i] - alpha * v[i];
    q[i] = qi;
    t[i] = u[i] + qi;
  }
}

// CG and CGS: x += alpha d; r -= alpha w; per block (r, r)
__global__ void __launch_bounds__(kBS) k_xr_update(int64_t n, double* __restrict__ x, const double* __restrict__ d,
                                                   double* __restrict__ r, const double* __restrict__ w,
                                                   const KrylovScalars* ks, double* __restrict__ part) {
  __shared__ double s_red[kBS / 64];
  if (ks->done) return;
  const double alpha = ks->alpha;
  double rr = 0.0;
  for (int64_t i = (int64_t)blockIdx.x * kBS + threadIdx.x; i < n; i += (int64_t)gridDim.x * kBS) {
    x[i] += alpha * d[i];
    const double ri = r[i] - alpha * w[i];
    r[i] = ri;
    rr += ri * ri;
  }
  rr = dev::block_sum<kBS>(rr, s_red);
  if (threadIdx.x == 0) part[2 * blockIdx.x] = rr;
}

// BiCGSTAB: p = r + beta (p - omega v)
__global__ void __launch_bounds__(kBS) k_bicg_p(int64_t n, const double* __restrict__ r, const double* __restrict__ v,
                                                double* __restrict__ p, const KrylovScalars* ks) {
  if (ks->done) return;
  const double beta = ks->beta, omega = ks->aux[0];
  for (int64_t i = (int64_t)blockIdx.x * kBS + threadIdx.x; i < n; i += (int64_t)gridDim.x * kBS)
    p[i] = r[i] + beta * (p[i] - omega * v[i]);
}

// BiCGSTAB: s = r - alpha v; per block (s, s)
__global__ void __launch_bounds__(kBS) k_bicg_s(int64_t n, const double* __restrict__ r, const double* __restrict__ v,
                                                double* __restrict__ s, const KrylovScalars* ks,
                                                double* __restrict__ part) {
  __shared__ double s_red[kBS / 64];
  if (ks->done) return;
  const double alpha = ks->alpha;
  double ss = 0.0;
  for (int64_t i = (int64_t)blockIdx.x * kBS + threadIdx.x; i < n; i += (int64_t)gridDim.x * kBS) {
    const double si = r[i] - alpha * v[i];
    s[i] = si;
    ss += si * si;
  }
  ss = dev::block_sum<kBS>(ss, s_red);
  if (threadIdx.x == 0) part[2 * blockIdx.x] = ss;
}

// BiCGSTAB: x += alpha ph + omega sh; r = s - omega t; per block (r, r). Once s met
// the tolerance only x += alpha ph is applied.
__global__ void __launch_bounds__(kBS) k_bicg_x(int64_t n, double* __restrict__ x, const double* __restrict__ ph,
                                                const double* __restrict__ sh, double* __restrict__ r,
                                                const double* __restrict__ s, const double* __restrict__ t,
                                                const KrylovScalars* ks, double* __restrict__ part) {
  __shared__ double s_red[kBS / 64];
  if (ks->done) return;
  const double alpha = ks->alpha, omega = ks->aux[0];
  const bool sconv = ks->aux[3] != 0.0;
  double rr = 0.0;
  for (int64_t i = (int64_t)blockIdx.x * kBS + threadIdx.x; i < n; i += (int64_t)gridDim.x * kBS) {
    if (sconv) {
      x[i] += alpha * ph[i];
    } else {
      x[i] += alpha * ph[i] + omega * sh[i];
      const double ri = s[i] - omega * t[i];
      r[i] = ri;
      rr += ri * ri;
    }
  }
  rr = dev::block_sum<kBS>(rr, s_red);
  if (threadIdx.x == 0) part[2 * blockIdx.x] = rr;
}

// CG: p = z + beta p (beta = 0 copies z)
__global__ void __launch_bounds__(kBS) k_cg_p(int64_t n, const double* __restrict__ z, double* __restrict__ p,
                                              const KrylovScalars* ks, int first) {
  if (ks->done) return;
  const double beta = first ? 0.0 : ks->beta;
  for (int64_t i = (int64_t)blockIdx.x * kBS + threadIdx.x; i < n; i += (int64_t)gridDim.x * kBS)
    p[i] = first ? z[i] : z[i] + beta * p[i];
}

__global__ void __launch_bounds__(kBS) k_jacobi_apply(int64_t n, const double* __restrict__ dinv,
                                                      const double* __restrict__ in, double* __restrict__ out,
                                                      const KrylovScalars* ks) {
  if (ks->done) return;
  for (int64_t i = (int64_t)blockIdx.x * kBS + threadIdx.x; i < n; i += (int64_t)gridDim.x * kBS)
    out[i] = dinv[i] * in[i];
}

// ---- SSOR sweeps
constexpr int kRunBS = 1024;
constexpr int kPieceRows = 512;
constexpr int kPieceEntries = 4 * (kRunBS - kPieceRows);
constexpr int kWindow = 8192;  // positions kept in LDS (64 KB)

// Time of a level in 1/30 us: in a one-block run, a piece takes 1 us and 1/30 us for every
// entry of its longest row; a launch takes its latency, more with long rows, most when all
// rows are long; and a run that starts anew fills its pipeline. Measured with all levels
// alike, in a run and launched: 256 rows of 4 entries 1.0 and 3.7 us; 1,024 of 4, 8, 16,
// 32, 64: 2.7 and 4.0, 4.9 and 6.1, 12.7 and 12.4, 37 and 31, 105 and 65; 2,048 of 4, 8,
// 16: 5.4 and 4.6, 9.5 and 6.8, 25 and 11. On octrees (rows of 3.5, the longest 9 to 13)
// a plan found so is as fast, within 1%, as runs of levels of up to 2,048 rows.
constexpr int64_t piece_cost(int64_t longest) { return 30 + longest; }
constexpr int64_t launch_cost(int64_t rows, int64_t entries, int64_t longest) {
  return std::max(100 + 6 * longest, 28 * entries / rows - 45);
}
constexpr int64_t kRunStart = 150;

// One triangle in level order: position k has the entries ptr[k] .. ptr[k + 1).
struct Sweep {
  const int32_t* ptr;
  const int32_t* col;   // neighbour's position
  const double* val;    // forward: omega a_ij; backward: a_ij
  const double* dinv;
  const double* own;    // forward: r_i; backward: y_i
  double* z;
  // launched levels alone: own value of position k is src[at[k]], and the result also goes
  // to out[row[k]] (if out is not null)
  const double* src;
  const int32_t* at;
  double* out;
  const int32_t* row;
};

template <bool FWD>
__device__ __forceinline__ double ssor_add(double t, double p) {
  return FWD ? t - p : t + p;
}
template <bool FWD>
__device__ __forceinline__ double ssor_finish(double t, double own, double dinv, double w) {
  return FWD ? t * dinv : own - (w * t) * dinv;
}

// A level as one launch: forward z_i = (r_i - sum_{j<i} (w a_ij) z_j) d_i^-1, backward
// z_i = y_i - (w sum_{j>i} a_ij z_j) d_i^-1. ALONE: at most kAlone levels and none in a run;
// the gathers into and out of level order are then part of the levels. Three launches
// fewer an application, but an index more in each level: an iteration of CGS, without and
// with it, 2 levels of 100,000 rows 94 and 85 us, 5 of 20,000 143 and 137, 10 of 100,000
// 415 and 413, 20 of 20,000 485 and 511.
constexpr size_t kAlone = 8;
template <bool FWD, bool ALONE>
__global__ void __launch_bounds__(kBS) k_ssor_level(Sweep S, int first, int end, double w, const KrylovScalars* ks) {
  if (ks->done) return;
  const int k = first + (int)(blockIdx.x * kBS + threadIdx.x);
  if (k >= end) return;
  const double own = ALONE ? S.src[S.at[k]] : S.own[k];
  double t = FWD ? own : 0.0;
  for (int32_t e = S.ptr[k], ee = S.ptr[k + 1]; e < ee; ++e) t = ssor_add<FWD>(t, S.val[e] * S.z[S.col[e]]);
  const double z = ssor_finish<FWD>(t, own, S.dinv[k], w);
  S.z[k] = z;
  if (ALONE && S.out) S.out[S.row[k]] = z;
}

struct RunLds {
  double z[kWindow];
  struct {
    double val[kPieceEntries];
    int32_t col[kPieceEntries];
  } piece[2];
};
static_assert(sizeof(RunLds) <= 160 * 1024, "one block's LDS");

// The pieces [i0, i1) of a run in one block, a barrier between pieces. Threads
// 0 .. kPieceRows - 1 solve piece i, a row each, from one LDS buffer, while the others
// write the entries of piece i + 1 to the other buffer; all loads are issued two to six
// pieces ahead. Neighbours within the last kWindow positions come from LDS; for an older
// one (or one of an earlier launch) the entry's value is replaced by its product when
// the entry is written (column -1), with a value loaded past the L1 two pieces before.
// It is in memory by then: at least 16 - 3 pieces old, and every solving wave completes
// all its stores every 8 pieces.
//
// Every load is unconditional (addresses clamped, into at least one entry): the compiler
// can then count the loads in flight and wait for just those it needs. A sweep over the 255,000-row mesh
// took 2.3 ms with one launch per level; in one block 1.46 ms with guarded loads (each
// piece waited for all of them), 0.92 ms with clamped loads and every thread doing both
// jobs, 0.87 ms with loads one piece ahead of their use and 0.69 ms now, about 1 us a
// piece. What bounds it is the latency of a piece, not bandwidth (22 GB/s).
template <bool FWD>
__global__ void __launch_bounds__(kRunBS) k_ssor_run(Sweep S, const int2* __restrict__ pieces, int i0, int i1,
                                                     double w, const KrylovScalars* ks) {
  extern __shared__ char s_mem[];
  RunLds& L = *reinterpret_cast<RunLds*>(s_mem);
  static_assert(kWindow >= 16 * kPieceRows, "older values must have left the store queue");
  constexpr int kStagers = kRunBS - kPieceRows, kPer = kPieceEntries / kStagers;
  static_assert(kPer * kStagers == kPieceEntries && kStagers % 64 == 0 && kPieceRows % 64 == 0, "");
  if (ks->done) return;
  struct Bounds {
    int r0, r1, e0, e1;
  };
  auto bounds = [&](int i) {  // pieces past i1 are empty
    const int2 p = pieces[min(i, i1)], q = pieces[min(i + 1, i1)];  // first position and entry
    return Bounds{p.x, q.x, p.y, q.y};
  };
  // LDS writes are done at the barrier; loads in flight stay in flight
  auto barrier = [] { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); };
  Bounds b[7];  // pieces i .. i + 6
#pragma unroll
  for (int u = 0; u < 7; ++u) b[u] = bounds(i0 + u);
  auto next = [&](int i) {
#pragma unroll
    for (int u = 0; u < 6; ++u) b[u] = b[u + 1];
    b[6] = bounds(i);
  };

  if (threadIdx.x < kPieceRows) {
    const int t = threadIdx.x;
    struct Row {
      double own, dinv;
      int32_t off, end;
    } r[4];
    auto load = [&](const Bounds& o, Row& q) {
      const int k = max(min(o.r0 + t, o.r1 - 1), 0);
      q.own = S.own[k];
      q.dinv = S.dinv[k];
      q.off = S.ptr[k];
      q.end = S.ptr[k + 1];
    };
    // entries e .. e + N - 1 of a row that ends at ee, all LDS reads in flight together
    auto add = [&](auto n, double acc, int e, int ee, const auto& p) {
      constexpr int N = decltype(n)::value;
      int32_t c[N];
      double v[N], z[N];
#pragma unroll
      for (int u = 0; u < N; ++u) {
        const int at = max(min(e + u, ee - 1), 0);
        c[u] = p.col[at];
        v[u] = p.val[at];
      }
#pragma unroll
      for (int u = 0; u < N; ++u) z[u] = L.z[c[u] & (kWindow - 1)];
#pragma unroll
      for (int u = 0; u < N; ++u)
        if (e + u < ee) acc = ssor_add<FWD>(acc, c[u] < 0 ? v[u] : v[u] * z[u]);
      return acc;
    };
    auto solve = [&](const Bounds& o, const Row& q, const auto& p) {
      if (t >= o.r1 - o.r0) return;
      double acc = FWD ? q.own : 0.0;
      const int e = q.off - o.e0, ee = q.end - o.e0;
      // rows of a level are in the order of their counts: a wave's rows are mostly alike
      if (!__any(ee - e > 4)) acc = add(std::integral_constant<int, 4>(), acc, e, ee, p);
      else if (!__any(ee - e > 8)) acc = add(std::integral_constant<int, 8>(), acc, e, ee, p);
      else
        for (int x = e; __any(x < ee); x += 16) acc = add(std::integral_constant<int, 16>(), acc, x, ee, p);
      const double z = ssor_finish<FWD>(acc, q.own, q.dinv, w);
      const int k = o.r0 + t;
      L.z[k & (kWindow - 1)] = z;
      S.z[k] = z;
    };
#pragma unroll
    for (int u = 0; u < 4; ++u) load(b[u], r[u]);
    barrier();
    for (int i = i0; i < i1; i += 8) {
#pragma unroll
      for (int u = 0; u < 8; ++u) {
        solve(b[0], r[u & 3], L.piece[u & 1]);
        load(b[4], r[u & 3]);
        if (u == 7) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        barrier();
        next(i + u + 7);
      }
    }
  } else {
    const int t = threadIdx.x - kPieceRows;
    const int run0 = pieces[i0].x;
    int32_t col[8][kPer];  // loaded six pieces ahead,
    double val[4][kPer];   // four,
    double far[4][kPer];   // and three
    auto oldest = [&](const Bounds& q) { return max(run0, q.r1 - kWindow); };
    auto entry = [&](const Bounds& q, int u) { return max(min(q.e0 + u * kStagers + t, q.e1 - 1), 0); };
    auto load_col = [&](const Bounds& q, int32_t* c) {
#pragma unroll
      for (int u = 0; u < kPer; ++u) c[u] = S.col[entry(q, u)];
    };
    auto load_val = [&](const Bounds& q, double* v) {
#pragma unroll
      for (int u = 0; u < kPer; ++u) v[u] = S.val[entry(q, u)];
    };
    // lanes without an old neighbour read position 0: one request for all of them
    auto load_far = [&](const Bounds& q, const int32_t* c, double* f) {
      const int lo = oldest(q);
#pragma unroll
      for (int u = 0; u < kPer; ++u)
        f[u] = __hip_atomic_load(S.z + (c[u] < lo ? c[u] : 0), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    };
    auto store = [&](const Bounds& q, const int32_t* c, const double* v, const double* f, auto& p) {
      const int lo = oldest(q);
#pragma unroll
      for (int u = 0; u < kPer; ++u) {
        const int e = u * kStagers + t;
        if (e < q.e1 - q.e0) {
          const bool old = c[u] < lo;
          p.val[e] = old ? v[u] * f[u] : v[u];
          p.col[e] = old ? -1 : c[u];
        }
      }
    };
#pragma unroll
    for (int u = 0; u < 6; ++u) load_col(b[u], col[u]);
#pragma unroll
    for (int u = 0; u < 4; ++u) load_val(b[u], val[u]);
#pragma unroll
    for (int u = 0; u < 3; ++u) load_far(b[u], col[u], far[u]);
    store(b[0], col[0], val[0], far[0], L.piece[0]);
    barrier();
    for (int i = i0; i < i1; i += 8) {
#pragma unroll
      for (int u = 0; u < 8; ++u) {
        load_far(b[3], col[(u + 3) & 7], far[(u + 3) & 3]);
        load_val(b[4], val[u & 3]);
        load_col(b[6], col[(u + 6) & 7]);
        store(b[1], col[(u + 1) & 7], val[(u + 1) & 3], far[(u + 1) & 3], L.piece[(u + 1) & 1]);
        barrier();
        next(i + u + 7);
      }
    }
  }
}

// entries of a triangle in level order
template <bool FWD>
__global__ void __launch_bounds__(kBS) k_ssor_pack(int64_t n, const int32_t* __restrict__ row,
                                                   const int32_t* __restrict__ rowptr,
                                                   const int32_t* __restrict__ diag, const int32_t* __restrict__ ccol,
                                                   const double* __restrict__ cval, const double* __restrict__ dinv,
                                                   const int32_t* __restrict__ pos, const int32_t* __restrict__ ptr,
                                                   double w, int32_t* __restrict__ col, double* __restrict__ val,
                                                   double* __restrict__ pdinv) {
  const int64_t k = (int64_t)blockIdx.x * kBS + threadIdx.x;
  if (k >= n) return;
  const int32_t i = row[k];
  pdinv[k] = dinv[i];
  const int32_t b = FWD ? rowptr[i] : diag[i] + 1, e = FWD ? diag[i] : rowptr[i + 1];
  const int32_t o = ptr[k];
  for (int32_t t = b; t < e; ++t) {
    col[o + t - b] = pos[ccol[t]];
    val[o + t - b] = FWD ? w * cval[t] : cval[t];
  }
}

// out[k] = in[idx[k]]: a vector into level order, from one sweep's order to the other's,
// or back to row order
__global__ void __launch_bounds__(kBS) k_ssor_gather(int64_t n, const int32_t* __restrict__ idx,
                                                     const double* __restrict__ in, double* __restrict__ out,
                                                     const KrylovScalars* ks) {
  if (ks->done) return;
  const int64_t k = (int64_t)blockIdx.x * kBS + threadIdx.x;
  if (k < n) out[k] = in[idx[k]];
}

// A triangle in level order: rows (by falling entry count within a level, so that a
// wave's rows are alike, then ascending), their positions, entry offsets, and the launches
// of a sweep, runs of pieces and single levels, by the least total of the costs above.
// cnt(i): entries of row i.
template <class Cnt>
void order_triangle(ngpb_ctx* c, ngpb_ctx::SsorTriangle& t, const std::vector<int32_t>& lev, int32_t nlev, Cnt&& cnt) {
  const size_t n = lev.size();
  std::vector<int32_t> first((size_t)nlev + 1, 0), rows(n), pos(n), ptr(n + 1, 0);
  for (int32_t l : lev) ++first[(size_t)l + 1];
  for (int32_t l = 0; l < nlev; ++l) first[(size_t)l + 1] += first[(size_t)l];
  std::vector<int32_t> fill(first.begin(), first.end() - 1);
  int32_t longest = 0;
  for (size_t i = 0; i < n; ++i) longest = std::max(longest, cnt(i));
  std::vector<int32_t> by_count(n), start((size_t)longest + 2, 0);
  for (size_t i = 0; i < n; ++i) ++start[(size_t)(longest - cnt(i)) + 1];
  for (int32_t q = 0; q <= longest; ++q) start[(size_t)q + 1] += start[(size_t)q];
  for (size_t i = 0; i < n; ++i) by_count[(size_t)start[(size_t)(longest - cnt(i))]++] = (int32_t)i;
  for (int32_t i : by_count) {
    const int32_t k = fill[(size_t)lev[(size_t)i]]++;
    rows[(size_t)k] = i;
    pos[(size_t)i] = k;
  }
  for (size_t k = 0; k < n; ++k) ptr[k + 1] = ptr[k] + cnt((size_t)rows[k]);
  auto piece_end = [&](int32_t k, int32_t b) {
    int32_t e = k;
    while (e < b && e - k < kPieceRows && ptr[(size_t)e + 1] - ptr[(size_t)k] <= kPieceEntries) ++e;
    return e;
  };
  // least cost up to each level with it in a run (0) or launched (1), and the choice before
  constexpr int64_t kNever = INT64_MAX / 4;
  std::vector<std::array<int8_t, 2>> from((size_t)nlev);
  int64_t cost[2] = {kRunStart, 0};  // before the first level: a run would start
  for (int32_t l = 0; l < nlev; ++l) {
    const int32_t a = first[(size_t)l], b = first[(size_t)l + 1];
    const int64_t row = cnt((size_t)rows[(size_t)a]);  // the longest: rows come by falling count
    int64_t in_run = kNever;
    // a row has to fit a piece; and without any entry in the whole triangle (a diagonal
    // operator) there is nothing to stage: k_ssor_run reads columns at clamped indices
    if (row <= kPieceEntries && longest > 0) {
      in_run = 0;
      for (int32_t k = a; k < b; k = piece_end(k, b)) in_run += piece_cost(cnt((size_t)rows[(size_t)k]));
    }
    const int64_t go_on = cost[0], start = cost[1] + kRunStart, either = std::min(cost[0], cost[1]);
    from[(size_t)l] = {(int8_t)(go_on <= start ? 0 : 1), (int8_t)(cost[0] < cost[1] ? 0 : 1)};
    cost[0] = std::min({go_on, start, kNever}) + in_run;
    cost[1] = either + launch_cost(b - a, ptr[(size_t)b] - ptr[(size_t)a], row);
  }
  std::vector<int8_t> launched((size_t)nlev);
  for (int32_t l = nlev - 1, s = cost[0] < cost[1] ? 0 : 1; l >= 0; s = from[(size_t)l][(size_t)s], --l)
    launched[(size_t)l] = (int8_t)s;
  t.runs.clear();
  std::vector<int32_t> pieces;
  for (int32_t l = 0; l < nlev; ++l) {
    const int32_t a = first[(size_t)l], b = first[(size_t)l + 1];
    if (launched[(size_t)l]) {
      t.runs.push_back({a, b, false});
      continue;
    }
    if (t.runs.empty() || !t.runs.back().pieces) {
      t.runs.push_back({(int32_t)pieces.size(), (int32_t)pieces.size(), true});
      pieces.push_back(a);
    }
    for (int32_t k = a; k < b;) pieces.push_back(k = piece_end(k, b));  // an end, the start of the next
    t.runs.back().last = (int32_t)pieces.size() - 1;
  }
  t.rows.upload(rows.data(), n, c->stream);
  t.pos.upload(pos.data(), n, c->stream);
  t.ptr.upload(ptr.data(), n + 1, c->stream);
  std::vector<int2> starts;
  for (int32_t k : pieces) starts.push_back(make_int2(k, ptr[(size_t)k]));
  t.pieces.upload(starts.data(), starts.size(), c->stream);
  t.col.resize((size_t)std::max(ptr[n], 1));
  t.val.resize((size_t)std::max(ptr[n], 1));
  t.dinv.resize(n);
  t.own.resize(n);
  t.z.resize(n);
  NGPB_HIP(hipStreamSynchronize(c->stream));  // the host arrays end here
}

}  // namespace

// Level sets of the SSOR sweeps and the diagonal positions, from the CSR pattern.
void build_ssor_levels(ngpb_ctx* c) {
  const int64_t n = c->n, nnz = c->nnz;
  std::vector<int32_t> rp((size_t)n + 1), col((size_t)nnz);
  c->rowptr.download(rp.data(), rp.size(), c->stream);
  c->col.download(col.data(), col.size(), c->stream);
  NGPB_HIP(hipStreamSynchronize(c->stream));
  std::vector<int32_t> diag((size_t)n), lf((size_t)n, 0), lb((size_t)n, 0);
  int32_t nf = 0, nb = 0;
  for (int64_t i = 0; i < n; ++i) {
    const int32_t* b = col.data() + rp[(size_t)i];
    const int32_t* e = col.data() + rp[(size_t)i + 1];
    const int32_t* d = std::lower_bound(b, e, (int32_t)i);
    NGPB_REQUIRE(d != e && *d == i, NGPB_E_NUMERIC, "operator has a row without a diagonal entry");
    diag[(size_t)i] = (int32_t)(d - col.data());
    int32_t l = 0;
    for (const int32_t* k = b; k < d; ++k) l = std::max(l, lf[(size_t)*k] + 1);
    lf[(size_t)i] = l;
    nf = std::max(nf, l + 1);
  }
  for (int64_t i = n - 1; i >= 0; --i) {
    int32_t l = 0;
    for (int32_t k = diag[(size_t)i] + 1; k < rp[(size_t)i + 1]; ++k) l = std::max(l, lb[(size_t)col[(size_t)k]] + 1);
    lb[(size_t)i] = l;
    nb = std::max(nb, l + 1);
  }
  order_triangle(c, c->ssor_f, lf, nf, [&](size_t i) { return diag[i] - rp[i]; });
  order_triangle(c, c->ssor_b, lb, nb, [&](size_t i) { return rp[i + 1] - diag[i] - 1; });
  {  // the backward sweep takes the forward sweep's result from the forward positions
    std::vector<int32_t> rows((size_t)n), pos((size_t)n), from((size_t)n);
    c->ssor_b.rows.download(rows.data(), rows.size(), c->stream);
    c->ssor_f.pos.download(pos.data(), pos.size(), c->stream);
    NGPB_HIP(hipStreamSynchronize(c->stream));
    for (size_t k = 0; k < from.size(); ++k) from[k] = pos[(size_t)rows[k]];
    c->ssor_b.from.upload(from.data(), from.size(), c->stream);
    c->diag_pos.upload(diag.data(), diag.size(), c->stream);
    NGPB_HIP(hipStreamSynchronize(c->stream));
  }
  c->have_levels = true;
}

namespace {

// One sweep over the runs of a triangle: its input is src[at[k]] at position k, t.z takes
// its result, and so does out in row order, if it is not null.
template <bool FWD>
void sweep(ngpb_ctx* c, const ngpb_ctx::SsorTriangle& t, double w, const double* src, const int32_t* at, double* out) {
  const bool alone = t.runs.size() <= kAlone && std::none_of(t.runs.begin(), t.runs.end(), [](const auto& r) { return r.pieces; });
  const Sweep S{t.ptr.p, t.col.p, t.val.p, t.dinv.p, t.own.p, t.z.p, src, at, out, t.rows.p};
  const dim3 G(blocks_for(c->n, kBS)), B(kBS);
  if (!alone) hipLaunchKernelGGL(k_ssor_gather, G, B, 0, c->stream, c->n, at, src, t.own.p, c->ks.p);
  for (const auto& r : t.runs) {
    if (alone)
      hipLaunchKernelGGL((k_ssor_level<FWD, true>), dim3(blocks_for(r.last - r.first, kBS)), dim3(kBS), 0, c->stream, S,
                         r.first, r.last, w, c->ks.p);
    else if (r.pieces)
      hipLaunchKernelGGL(k_ssor_run<FWD>, dim3(1), dim3(kRunBS), sizeof(RunLds), c->stream, S, t.pieces.p, r.first,
                         r.last, w, c->ks.p);
    else
      hipLaunchKernelGGL((k_ssor_level<FWD, false>), dim3(blocks_for(r.last - r.first, kBS)), dim3(kBS), 0, c->stream, S,
                         r.first, r.last, w, c->ks.p);
  }
  if (!alone && out) hipLaunchKernelGGL(k_ssor_gather, G, B, 0, c->stream, c->n, t.pos.p, t.z.p, out, c->ks.p);
}

// The packed entries of one triangle for the current values and relaxation.
template <bool FWD>
void pack_triangle(ngpb_ctx* c, ngpb_ctx::SsorTriangle& t, double w) {
  hipLaunchKernelGGL(k_ssor_pack<FWD>, dim3(blocks_for(c->n, kBS)), dim3(kBS), 0, c->stream, c->n, t.rows.p,
                     c->rowptr.p, c->diag_pos.p, c->col.p, c->val.p, c->dinv.p, t.pos.p, t.ptr.p, w, t.col.p, t.val.p,
                     t.dinv.p);
  NGPB_HIP(hipGetLastError());
  NGPB_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(k_ssor_run<FWD>),
                               hipFuncAttributeMaxDynamicSharedMemorySize, sizeof(RunLds)));
}

// z = M^-1 in; returns the vector that holds the result (`in` itself without a
// preconditioner). c->dinv must hold the inverse diagonal.
const double* psolve(ngpb_ctx* c, int precon, double w, const double* in, double* out) {
  const int64_t n = c->n;
  const KrylovScalars* ks = c->ks.p;
  if (precon == NGPB_PRECON_NONE) return in;
  if (precon == NGPB_PRECON_JACOBI) {
    hipLaunchKernelGGL(k_jacobi_apply, dim3(vec_grid(n)), dim3(kBS), 0, c->stream, n, c->dinv.p, in, out, ks);
    return out;
  }
  sweep<true>(c, c->ssor_f, w, in, c->ssor_f.rows.p, nullptr);
  sweep<false>(c, c->ssor_b, w, c->ssor_f.z.p, c->ssor_b.from.p, out);
  return out;
}

void prepare_precon(ngpb_ctx* c, int precon, double w) {
  if (precon != NGPB_PRECON_SSOR) return;
  if (!c->have_levels) build_ssor_levels(c);
  pack_triangle<true>(c, c->ssor_f, w);
  pack_triangle<false>(c, c->ssor_b, w);
}

}  // namespace

double ssor_omega(const ngpb_solve_opts& o) { return o.omega > 0.0 ? o.omega : 1.0; }

void check_lis_options(const ngpb_solve_opts& o) {
  NGPB_REQUIRE(o.solver == NGPB_SOLVER_CG || o.solver == NGPB_SOLVER_CGS || o.solver == NGPB_SOLVER_BICGSTAB,
               NGPB_E_ARG, "solver must be CG, CGS or BiCGSTAB");
  NGPB_REQUIRE(o.precon == NGPB_PRECON_JACOBI || o.precon == NGPB_PRECON_NONE || o.precon == NGPB_PRECON_SSOR,
               NGPB_E_ARG, "preconditioner must be Jacobi, none or SSOR");
  NGPB_REQUIRE(o.precon != NGPB_PRECON_SSOR || (ssor_omega(o) > 0.0 && ssor_omega(o) < 2.0), NGPB_E_ARG,
               "SSOR relaxation must lie in (0, 2)");
}

void precond_apply(ngpb_ctx* c, int precon, double omega, const double* r, double* z) {
  check_operator(c);  // inverse diagonal, NaN/Inf and diagonal checks
  prepare_precon(c, precon, omega);
  ensure_reduce(c, 2048);
  KrylovScalars zero;
  std::memset(&zero, 0, sizeof(zero));
  NGPB_HIP(hipMemcpyAsync(c->ks.p, &zero, sizeof(zero), hipMemcpyHostToDevice, c->stream));
  const double* res = psolve(c, precon, omega, r, z);
  if (res != z) NGPB_HIP(hipMemcpyAsync(z, res, (size_t)c->n * sizeof(double), hipMemcpyDeviceToDevice, c->stream));
  NGPB_HIP(hipGetLastError());
  NGPB_HIP(hipStreamSynchronize(c->stream));
}

void solve_lis(ngpb_ctx* c, const ngpb_solve_opts& o, ngpb_solve_stats& st) {
  check_lis_options(o);
  const int64_t n = c->n;
  const double w = ssor_omega(o);
  const void* rec = slice_records(c, nullptr);
  prepare_precon(c, o.precon, w);
  c->x.resize((size_t)n);
  c->r.resize((size_t)n);
  c->z.reserve((size_t)n);
  c->p.reserve((size_t)n);
  c->q.reserve((size_t)n);
  for (auto* b : {&c->lis_rt, &c->lis_u, &c->lis_v, &c->lis_ph, &c->lis_uh, &c->lis_t}) b->reserve((size_t)n);
  const unsigned gv = vec_grid(n);
  const int64_t gs_region = std::max<int64_t>(spmv_fp64_grid(c, rec), 2048);
  ensure_reduce(c, gs_region + 2 * (int64_t)gv);
  double* spart = c->red.partials.p;             // SpMV (x, y) partials, stride 1
  double* dpart = c->red.partials.p + gs_region;  // vector partials, stride 2
  KrylovScalars* ks = c->ks.p;
  double *x = c->x.p, *r = c->r.p, *p = c->p.p, *q = c->q.p, *z = c->z.p;
  double *rt = c->lis_rt.p, *u = c->lis_u.p, *v = c->lis_v.p, *ph = c->lis_ph.p, *uh = c->lis_uh.p, *t = c->lis_t.p;
  const dim3 G(gv), B(kBS), F(1), BF(kFin);
  const int np = (int)gv, nsp = (int)spmv_fp64_grid(c, rec);
  auto fin = [&](const double* part, int cnt, int stride, int what) {
    hipLaunchKernelGGL(k_lis_fin, F, BF, 0, c->stream, ks, part, cnt, stride, what, o.solver);
  };
  hipEvent_t e0, e1;
  NGPB_HIP(hipEventCreate(&e0));
  NGPB_HIP(hipEventCreate(&e1));
  NGPB_HIP(hipEventRecord(e0, c->stream));
  hipLaunchKernelGGL(k_lis_init, G, B, 0, c->stream, n, c->rhs.p, x, r, rt, p, q, v, dpart);
  hipLaunchKernelGGL(k_lis_fin_init, F, BF, 0, c->stream, ks, dpart, np, o.tol * o.tol, o.maxiter);
  if (o.solver == NGPB_SOLVER_CG) {
    const double* zz = psolve(c, o.precon, w, r, z);
    hipLaunchKernelGGL(k_dots<false>, G, B, 0, c->stream, n, r, zz, nullptr, nullptr, ks, dpart);
    fin(dpart, np, 2, kFinCgRho0);
    hipLaunchKernelGGL(k_cg_p, G, B, 0, c->stream, n, zz, p, ks, 1);
  }
  NGPB_HIP(hipGetLastError());
  const int chunk = std::max(1, o.check_every);
  while (true) {
    for (int k = 0; k < chunk; ++k) {
      if (o.solver == NGPB_SOLVER_CG) {
        spmv_fp64_dot(c, p, q, spart, rec);  // q = A p with (p, q) partials
        fin(spart, nsp, 1, kFinAlpha);
        hipLaunchKernelGGL(k_xr_update, G, B, 0, c->stream, n, x, p, r, q, ks, dpart);
        fin(dpart, np, 2, kFinResid);
        const double* zz = psolve(c, o.precon, w, r, z);
        hipLaunchKernelGGL(k_dots<false>, G, B, 0, c->stream, n, r, zz, nullptr, nullptr, ks, dpart);
        fin(dpart, np, 2, kFinCgBeta);
        hipLaunchKernelGGL(k_cg_p, G, B, 0, c->stream, n, zz, p, ks, 0);
      } else if (o.solver == NGPB_SOLVER_CGS) {
        hipLaunchKernelGGL(k_dots<false>, G, B, 0, c->stream, n, rt, r, nullptr, nullptr, ks, dpart);
        fin(dpart, np, 2, kFinRho);
        hipLaunchKernelGGL(k_cgs_up, G, B, 0, c->stream, n, r, q, u, p, ks);
        const double* pp = psolve(c, o.precon, w, p, ph);
        spmv_fp64_dot(c, pp, v, spart, rec);
        hipLaunchKernelGGL(k_dots<false>, G, B, 0, c->stream, n, rt, v, nullptr, nullptr, ks, dpart);
        fin(dpart, np, 2, kFinAlpha);
        hipLaunchKernelGGL(k_cgs_q, G, B, 0, c->stream, n, u, v, q, t, ks);
        const double* uu = psolve(c, o.precon, w, t, uh);
        spmv_fp64_dot(c, uu, ph, spart, rec);  // A uh into ph, free once v = A ph was formed
        hipLaunchKernelGGL(k_xr_update, G, B, 0, c->stream, n, x, uu, r, ph, ks, dpart);
        fin(dpart, np, 2, kFinResid);
      } else {  // BiCGSTAB; s lives in u, its preconditioned copy in uh
        hipLaunchKernelGGL(k_dots<false>, G, B, 0, c->stream, n, rt, r, nullptr, nullptr, ks, dpart);
        fin(dpart, np, 2, kFinRho);
        hipLaunchKernelGGL(k_bicg_p, G, B, 0, c->stream, n, r, v, p, ks);
        const double* pp = psolve(c, o.precon, w, p, ph);
        spmv_fp64_dot(c, pp, v, spart, rec);
        hipLaunchKernelGGL(k_dots<false>, G, B, 0, c->stream, n, rt, v, nullptr, nullptr, ks, dpart);
        fin(dpart, np, 2, kFinAlpha);
        hipLaunchKernelGGL(k_bicg_s, G, B, 0, c->stream, n, r, v, u, ks, dpart);
        fin(dpart, np, 2, kFinBicgS);
        const double* ss = psolve(c, o.precon, w, u, uh);
        spmv_fp64_dot(c, ss, t, spart, rec);
        hipLaunchKernelGGL(k_dots<true>, G, B, 0, c->stream, n, t, u, t, t, ks, dpart);
        fin(dpart, np, 2, kFinOmega);
        hipLaunchKernelGGL(k_bicg_x, G, B, 0, c->stream, n, x, pp, ss, r, u, t, ks, dpart);
        fin(dpart, np, 2, kFinBicgResid);
      }
    }
    NGPB_HIP(hipGetLastError());
    NGPB_HIP(hipMemcpyAsync(c->ks_host, ks, sizeof(KrylovScalars), hipMemcpyDeviceToHost, c->stream));
    NGPB_HIP(hipStreamSynchronize(c->stream));
    if (c->ks_host->done) break;
  }
  NGPB_HIP(hipEventRecord(e1, c->stream));
  NGPB_HIP(hipEventSynchronize(e1));
  float ms = 0.f;
  NGPB_HIP(hipEventElapsedTime(&ms, e0, e1));
  (void)hipEventDestroy(e0);
  (void)hipEventDestroy(e1);
  const KrylovScalars& h = *c->ks_host;
  st.status = h.status;
  st.iterations = h.iter;
  st.replacements = 0;
  st.relres = h.bb > 0 ? std::sqrt(h.rr / h.bb) : 0.0;
  st.ms_solve = ms;
  // matrix-vector products and preconditioner applications of one iteration, plus
  // the vector streams (8 bytes each)
  const double spmv = spmv_fp64_bytes(c);
  const double pre = o.precon == NGPB_PRECON_SSOR ? spmv + (double)n * 8.0 * 3.0
                     : o.precon == NGPB_PRECON_JACOBI ? (double)n * 24.0 : 0.0;
  const double vec = o.solver == NGPB_SOLVER_CG ? 14.0 : o.solver == NGPB_SOLVER_CGS ? 22.0 : 24.0;
  const double nmv = o.solver == NGPB_SOLVER_CG ? 1.0 : 2.0;
  st.bytes_per_iter = nmv * (spmv + pre) + (double)n * 8.0 * vec;
  c->have_phi = true;
  c->phi_len = c->n;
}

}  // namespace ngpb
