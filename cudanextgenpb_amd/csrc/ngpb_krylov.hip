// FP64 CSR SpMV and the plain Jacobi-preconditioned CG (LIS -i cg -p jacobi as
// called from lis_compute_electric_potential, src/pb_class.cpp:2243-2329).
//
// SpMV: a block of 256 threads owns 256 consecutive rows. Their column indices and
// values are read once, coalesced, and each (value, x[column]) pair is staged in
// LDS; each thread then forms its row sum in column order as a chain of fused
// multiply-adds starting from zero (the same arithmetic as the oracle's SpMV, so the
// results are bit-identical). Blocks whose rows hold more than kCap entries stage
// them in pieces of kCap, each row carrying its chain from piece to piece (reading
// such blocks' entries row by row from global memory instead made the 8.04M-row
// SpMV 10% slower: 217 against 195 us).
//
// CG iteration, three kernels: SpMV + per-block (p, q) -> x/r update + per-block
// (r, D^-1 r), (r, r) -> stop test and new direction. Each kernel first combines the
// previous kernel's per-block partial sums itself, every block in the same fixed
// order, so all blocks hold identical scalars; reductions are deterministic and no
// kernel needs a device-wide memory fence (on a multi-XCD GPU an agent-scope fence
// writes back the XCD's L2, which would serialize every block). Scalars live in
// device memory; the host polls the stop flag every `check_every` iterations and
// kernels launched after the stop exit at once.
#include <algorithm>
#include <chrono>
#include <cmath>
#include <cstring>
#include <mutex>

#include "ngpb_internal.h"

namespace ngpb {
namespace {

constexpr int kBS = 256;
constexpr int kCap = 2048;  // staged entries per block
constexpr int kFin = 1024;  // finalize block size

// SCHED 0: block b takes chunks b, b + G, ...; SCHED 1: block b takes one contiguous
// range of chunks, with blocks renumbered so that the blocks on one XCD (block id
// mod 8) cover one contiguous eighth of the rows (L2 reuse of the x gathers); the
// grid is then the number of blocks resident at once.
template <bool DOT, int SCHED>
__global__ void __launch_bounds__(kBS) k_spmv64(int64_t n, const int32_t* __restrict__ rowptr,
                                                 const int32_t* __restrict__ col, const double* __restrict__ val,
                                                 const double* __restrict__ x, double* __restrict__ y,
                                                 const KrylovScalars* ks, double* __restrict__ partials) {
  __shared__ double s_val[kCap];
  __shared__ double s_x[kCap];
  __shared__ double s_red[kBS / 64];
  if (DOT && ks->done) return;
  double part = 0.0;
  const int64_t nchunks = (n + kBS - 1) / kBS;
  int64_t c_begin = blockIdx.x, c_end = nchunks, c_step = gridDim.x;
  if (SCHED == 1) {
    const unsigned nb = gridDim.x, b = blockIdx.x;
    const int64_t lb = (nb % 8u == 0u) ? (int64_t)((b % 8u) * (nb / 8u) + b / 8u) : (int64_t)b;
    c_begin = lb * nchunks / nb;
    c_end = (lb + 1) * nchunks / nb;
    c_step = 1;
  }
  for (int64_t chunk = c_begin; chunk < c_end; chunk += c_step) {
    const int64_t r0 = chunk * kBS;
    const int64_t r1 = min(r0 + kBS, n);
    const int64_t row = r0 + threadIdx.x;
    const int64_t e0 = rowptr[r0], e1 = rowptr[r1];
    const int64_t rb = row < n ? (int64_t)rowptr[row] : e1, re = row < n ? (int64_t)rowptr[row + 1] : e1;
    double sum = 0.0;
    // the chunk's entries staged kCap at a time; each row continues its fma chain
    // across pieces, so the order of its terms is the column order as before
    for (int64_t p0 = e0; p0 < e1; p0 += kCap) {
      const int64_t p1 = min(p0 + (int64_t)kCap, e1);
      __syncthreads();  // the previous piece's rows are done with the staging buffers
      // all loads of the piece are issued before any is used: indices past the piece's
      // last entry are clamped to it and their LDS slots are never read
      constexpr int kU = kCap / kBS;
      double v[kU];
      int c[kU];
      const int64_t kl = p1 - 1;
#pragma unroll
      for (int u = 0; u < kU; ++u) {
        const int64_t k = min(p0 + threadIdx.x + (int64_t)u * kBS, kl);
        // the matrix is read once per SpMV: non-temporal loads leave the last-level cache
        // to the CG vectors (FP64 solve of the 8M-unknown globular system 174 -> 170 ms)
        v[u] = __builtin_nontemporal_load(&val[k]);
        c[u] = __builtin_nontemporal_load(&col[k]);
      }
#pragma unroll
      for (int u = 0; u < kU; ++u) {
        const int64_t k = p0 + threadIdx.x + (int64_t)u * kBS;
        s_val[k - p0] = v[u];
        s_x[k - p0] = x[c[u]];
      }
      __syncthreads();
      const int64_t kb = max(rb, p0), ke = min(re, p1);
      for (int64_t k = kb; k < ke; ++k) sum = fma(s_val[k - p0], s_x[k - p0], sum);
    }
    if (row < n) y[row] = sum;
    if (DOT && row < n) part += x[row] * sum;
  }
  if (DOT) {
    part = dev::block_sum<kBS>(part, s_red);
    if (threadIdx.x == 0) partials[blockIdx.x] = part;
  }
}

// ---- slice records
// Most rows of a mesh operator belong to 64-row slices whose entries lie on a few
// diagonals (column - row), with the same value along a diagonal wherever the medium is
// uniform. A record lists a slice's diagonals in ascending order, which rows have an
// entry there and, unless it varies, the value: the product then reads 288 bytes of
// record and contiguous runs of x instead of 12 bytes per entry. Values that vary are
// read from the CSR, and slices with more diagonals are staged as in k_spmv64. Every row
// still sums its entries in column order, so the results are the same bit for bit.
constexpr int kDiags = 14;
// Most rows of k_pcg_block. Whole solves of uniform grids: 4,096 rows 1,340 us with three
// launches per iteration, 822 in one block; 512 rows 863 and 239; 8,000 rows 1,774 and
// 1,708 (8 rows per thread, which spill), so the line lies at 4 rows per thread.
constexpr int kBlockRows = 4096;
// and most diagonals over all its slices (nine each at 4,096 rows): an iteration takes 2 us
// and 1/60 us for each of varying values (448: 9.2 us, 520: 10.7, 611: 12.8, 832: 15.9)
// against 11 to 14 us, by the host's pace, of three launches.
constexpr int kBlockDiags = 576;
struct SliceRec {
  int32_t count;  // diagonals, -1: more than kDiags
  uint32_t vary;  // bit k: diagonal k's values differ
  int32_t delta[kDiags];
  uint64_t rows[kDiags];  // bit per row
  double val[kDiags];
};
static_assert(sizeof(SliceRec) == 288, "SliceRec is 288 bytes");

// Whether the products of a system use its records: `staged` of its slices have none. Up
// to 2^18 rows a wave has one slice, and the slowest slice is the product: only without
// staged ones. From 2^19 rows on, where waves have several, up to two thirds of them, and
// in between the line runs straight. Per iteration with records and from the CSR alone:
// 27,000 rows, 18% staged: 13.9 and 12.3 us; 216,000, none: 17.0 and 18.2, 24%: 19.4 and
// 18.4; 421,875, 23%: 25.9 and 27.3, 69%: 28.5 and 27.4; 1 million, 58%: 44.5 and 47.4,
// 85%: 48.9 and 47.5. Rows without any pattern of 183 entries: 443 us a product and 285.
bool use_records(int64_t n, int64_t staged) {
  const int64_t lo = int64_t(1) << 18, slices = (n + 63) / 64;
  return 3 * lo * staged <= 2 * slices * std::clamp<int64_t>(n - lo, 0, lo);
}

// whether a system's CG runs in one block
bool use_block(int64_t n, int staged, int diags) { return n <= kBlockRows && !staged && diags <= kBlockDiags; }

// one wave per slice; flags[1] counts the slices with more than kDiags diagonals, flags[2]
// the diagonals of the others (at up to kBlockRows rows)
__global__ void __launch_bounds__(kBS) k_slice_rec(int64_t n, const int32_t* __restrict__ rowptr,
                                                   const int32_t* __restrict__ col, const double* __restrict__ val,
                                                   SliceRec* __restrict__ recs, int* __restrict__ flags) {
  const int64_t s = (int64_t)blockIdx.x * (kBS / 64) + (threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  const int64_t row = s * 64 + lane;
  int64_t e = 0, end = 0;
  if (row < n) {
    e = rowptr[row];
    end = rowptr[row + 1];
  }
  SliceRec& R = recs[s];
  int k = 0;
  uint32_t vary = 0;
  while (true) {
    int d = e < end ? (int)((int64_t)col[e] - row) : INT32_MAX;
    int m = d;
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) m = min(m, __shfl_xor(m, off, 64));
    if (m == INT32_MAX) break;
    if (k == kDiags) {
      k = -1;
      break;
    }
    const bool has = d == m;
    const uint64_t rows = __ballot(has);
    const double v = has ? val[e] : 0.0;
    const long long bits = __double_as_longlong(v);
    const long long first = __shfl(bits, __ffsll((unsigned long long)rows) - 1, 64);
    if (__ballot(has && bits != first)) vary |= 1u << k;
    if (lane == 0) {
      R.delta[k] = m;
      R.rows[k] = rows;
      R.val[k] = __longlong_as_double(first);
    }
    if (has) ++e;
    ++k;
  }
  if (lane == 0 && s * 64 < n) {
    R.count = k;
    R.vary = vary;
  }
  __shared__ int s_k[kBS / 64];
  if (lane == 0) s_k[threadIdx.x >> 6] = k;
  __syncthreads();
  if (threadIdx.x != 0) return;
  int staged = 0, diags = 0;
  for (int q = 0; q < kBS / 64; ++q) {
    staged += s_k[q] < 0 ? 1 : 0;
    diags += max(s_k[q], 0);
  }
  if (staged) atomicAdd(flags + 1, staged);
  if (n <= kBlockRows) atomicAdd(flags + 2, diags);
}

// k_spmv64 from slice records: the same rows per thread and the same partial sums. A
// record is read one word per lane, the next slice's while this one is worked on, and
// its fields are broadcast from there; kGo diagonals' loads of x are in flight together.
// Bound by the latency of record, x and store at one or two slices per wave. 1 million
// rows of a uniform grid: 26 us from the CSR, 12.4 with each field a scalar load when it
// is needed, 11.1 so; 2.1 million rows: 50, 24.2, 22.0 us.
template <int SCHED>
__global__ void __launch_bounds__(kBS) k_spmv64_rec(int64_t n, const int32_t* __restrict__ rowptr,
                                                     const int32_t* __restrict__ col, const double* __restrict__ val,
                                                     const SliceRec* __restrict__ recs, const double* __restrict__ x,
                                                     double* __restrict__ y, const KrylovScalars* ks,
                                                     double* __restrict__ partials) {
  constexpr int kWaveCap = 256, kGo = 7, kSW = kBS / 64;
  constexpr int kRows = 2 + kDiags, kVal = kRows + 2 * kDiags;  // words before the fields
  __shared__ double s_val[kSW * kWaveCap];
  __shared__ double s_x[kSW * kWaveCap];
  __shared__ double s_red[kSW];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  double part = 0.0;
  const int64_t nchunks = (n + kBS - 1) / kBS;
  int64_t c_begin = blockIdx.x, c_end = nchunks, c_step = gridDim.x;
  if (SCHED == 1) {
    const unsigned nb = gridDim.x, b = blockIdx.x;
    const int64_t lb = (nb % 8u == 0u) ? (int64_t)((b % 8u) * (nb / 8u) + b / 8u) : (int64_t)b;
    c_begin = lb * nchunks / nb;
    c_end = (lb + 1) * nchunks / nb;
    c_step = 1;
  }
  const int64_t nslices = (n + 63) / 64;
  const int32_t* const words = reinterpret_cast<const int32_t*>(recs);
  // words l and 64 + l of a record (72 in all; lanes 8.. repeat the last)
  auto word_at = [&](int64_t chunk, int w) {
    const int64_t s = min(min(chunk, nchunks - 1) * kSW + wave, nslices - 1);
    return words[s * 72 + min(w, 71)];
  };
  int n0 = word_at(c_begin, lane), n1 = word_at(c_begin, 64 + lane);
  if (ks->done) return;
  for (int64_t chunk = c_begin; chunk < c_end; chunk += c_step) {
    const int w0 = n0, w1 = n1;
    n0 = word_at(chunk + c_step, lane);
    n1 = word_at(chunk + c_step, 64 + lane);
    const int64_t s = __builtin_amdgcn_readfirstlane((int)(chunk * kSW + wave));
    if (s >= nslices) continue;
    const int64_t row = s * 64 + lane;
    auto word = [&](int k) {
      return (uint32_t)(k < 64 ? __builtin_amdgcn_readlane(w0, k) : __builtin_amdgcn_readlane(w1, k - 64));
    };
    auto pair = [&](int k) { return (uint64_t)word(k) | (uint64_t)word(k + 1) << 32; };
    const int count = (int)word(0);
    double sum = 0.0;
    if (count >= 0) {
      const uint32_t vary = word(1);
      int64_t e = vary && row < n ? (int64_t)rowptr[row] : 0;  // the row's next entry
      const int64_t safe = min(row, n - 1);
#pragma unroll
      for (int k0 = 0; k0 < kDiags; k0 += kGo) {
        if (k0 >= count) break;
        double xv[kGo], v[kGo];
        bool has[kGo];
#pragma unroll
        for (int u = 0; u < kGo; ++u) {
          const int k = k0 + u;
          has[u] = k < count && ((pair(kRows + 2 * k) >> lane) & 1);
          xv[u] = x[has[u] ? row + (int)word(2 + k) : safe];
          v[u] = __longlong_as_double((long long)pair(kVal + 2 * k));
        }
        if (vary) {
#pragma unroll
          for (int u = 0; u < kGo; ++u) {
            if (has[u] && ((vary >> (k0 + u)) & 1)) v[u] = val[e];
            if (has[u]) ++e;
          }
        }
#pragma unroll
        for (int u = 0; u < kGo; ++u)
          if (has[u]) sum = fma(v[u], xv[u], sum);
      }
    } else {
      // a slice of its own shape: its entries staged in the wave's part of the LDS
      const int64_t last = min(s * 64 + 63, n - 1);
      const int64_t e0 = rowptr[s * 64], e1 = rowptr[last + 1];
      const int64_t rb = row < n ? (int64_t)rowptr[row] : e1, re = row < n ? (int64_t)rowptr[row + 1] : e1;
      double* wv = s_val + wave * kWaveCap;
      double* wx = s_x + wave * kWaveCap;
      for (int64_t p0 = e0; p0 < e1; p0 += kWaveCap) {
        const int64_t p1 = min(p0 + (int64_t)kWaveCap, e1);
        constexpr int kU = kWaveCap / 64;
        double v[kU];
        int c[kU];
#pragma unroll
        for (int u = 0; u < kU; ++u) {
          const int64_t k = min(p0 + lane + u * 64, p1 - 1);
          v[u] = __builtin_nontemporal_load(&val[k]);
          c[u] = __builtin_nontemporal_load(&col[k]);
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();  // the previous piece has been read
#pragma unroll
        for (int u = 0; u < kU; ++u) {
          wv[lane + u * 64] = v[u];
          wx[lane + u * 64] = x[c[u]];
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
        const int64_t kb = max(rb, p0), ke = min(re, p1);
        for (int64_t k = kb; k < ke; ++k) sum = fma(wv[k - p0], wx[k - p0], sum);
      }
    }
    if (row < n) {
      y[row] = sum;
      part += x[row] * sum;
    }
  }
  part = dev::block_sum<kBS>(part, s_red);
  if (threadIdx.x == 0) partials[blockIdx.x] = part;
}

// ---- small systems: the whole CG in one block
// An iteration of three launches takes 11 us however few the rows: their latency. For at
// most kBlockRows rows, in slices that all have a record (own entry lists would be read
// from memory in every iteration: a 5,559-row octree operator took 3.7 ms for 1.8), one
// block keeps p and A p in LDS and r and 1 / diag of its R rows per thread in registers,
// and takes up to `steps` iterations per launch with three barriers each: 2.3 us per
// iteration at 512 rows, 6.3 at 4,096, where reading varying values is most of it.
constexpr int kBlk = 1024;

// sums of a and b over the block, in every thread; slot alternates between calls
__device__ __forceinline__ double2 blk_sum2(double a, double b, double2* slot) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) {
    a += __shfl_xor(a, off, 64);
    b += __shfl_xor(b, off, 64);
  }
  if ((threadIdx.x & 63) == 0) slot[threadIdx.x >> 6] = make_double2(a, b);
  __syncthreads();
  double2 t = make_double2(0.0, 0.0);
#pragma unroll
  for (int w = 0; w < kBlk / 64; ++w) {
    t.x += slot[w].x;
    t.y += slot[w].y;
  }
  return t;
}

// Aligned: the loop is fetched over and over by one CU, and where its code falls moved an
// iteration at 4,096 rows between 8.3 and 8.5 us.
template <int R>
__global__ void __launch_bounds__(kBlk) __attribute__((aligned(4096))) k_pcg_block(int n, const int32_t* __restrict__ rowptr, const double* __restrict__ val,
                                                     const SliceRec* __restrict__ recs, const double* __restrict__ dinv,
                                                     const double* __restrict__ b, double* __restrict__ x,
                                                     double* __restrict__ r, double* __restrict__ p, KrylovScalars* ks,
                                                     double tol2, int maxiter, int first, int steps) {
  constexpr int kGo = 7;
  __shared__ double s_p[R * kBlk], s_q[R * kBlk];
  __shared__ int s_e[R * kBlk];
  __shared__ double2 s_red[2][kBlk / 64];
  const int t = threadIdx.x, lane = t & 63;
  double xr[R], rr[R], di[R];
  double rho, stop_rr, RR = 0.0;
  int it = 0, done = 0, status = 0;
#pragma unroll
  for (int j = 0; j < R; ++j) s_e[j * kBlk + t] = j * kBlk + t < n ? rowptr[j * kBlk + t] : 0;
  if (first) {
    double rz = 0.0, bb = 0.0;
#pragma unroll
    for (int j = 0; j < R; ++j) {
      const int row = j * kBlk + t;
      const double bi = row < n ? b[row] : 0.0;
      di[j] = row < n ? dinv[row] : 0.0;
      const double zi = di[j] * bi;
      xr[j] = 0.0;
      rr[j] = bi;
      s_p[row] = zi;
      rz += bi * zi;
      bb += bi * bi;
    }
    const double2 S = blk_sum2(rz, bb, s_red[1]);
    rho = S.x;
    RR = S.y;
    stop_rr = tol2 * S.y;
    done = S.y == 0.0;
    if (t == 0) {
      ks->bb = S.y;
      ks->stop_rr = stop_rr;
    }
  } else {
    if (ks->done) return;
#pragma unroll
    for (int j = 0; j < R; ++j) {
      const int row = j * kBlk + t;
      xr[j] = row < n ? x[row] : 0.0;
      rr[j] = row < n ? r[row] : 0.0;
      di[j] = row < n ? dinv[row] : 0.0;
      s_p[row] = row < n ? p[row] : 0.0;
    }
    rho = ks->rho;
    stop_rr = ks->stop_rr;
    it = ks->iter;
    __syncthreads();
  }
  for (int k = 0; k < steps && !done; ++k) {
    double pq = 0.0;
#pragma unroll
    for (int j = 0; j < R; ++j) {
      const int s = __builtin_amdgcn_readfirstlane(j * (kBlk / 64) + (t >> 6));
      const int row = j * kBlk + t;
      if (s * 64 >= n) break;
      const SliceRec& S = recs[s];
      double sum = 0.0;
      const uint32_t vary = S.vary;
      int e = s_e[row];  // the row's next entry
#pragma unroll
      for (int k0 = 0; k0 < kDiags; k0 += kGo) {
        if (k0 >= S.count) break;
        double pv[kGo], v[kGo];
        bool has[kGo];
#pragma unroll
        for (int u = 0; u < kGo; ++u) {
          has[u] = k0 + u < S.count && ((S.rows[k0 + u] >> lane) & 1);
          pv[u] = s_p[has[u] ? row + S.delta[k0 + u] : row];
          v[u] = S.val[k0 + u];
        }
        if (vary) {
#pragma unroll
          for (int u = 0; u < kGo; ++u) {
            if (has[u] && ((vary >> (k0 + u)) & 1)) v[u] = val[e];
            if (has[u]) ++e;
          }
        }
#pragma unroll
        for (int u = 0; u < kGo; ++u)
          if (has[u]) sum = fma(v[u], pv[u], sum);
      }
      s_q[row] = sum;
      pq += s_p[row] * sum;  // rows past n: p and sum are 0
    }
    const double alpha = rho / blk_sum2(pq, 0.0, s_red[0]).x;
    double rz = 0.0, r2 = 0.0;
#pragma unroll
    for (int j = 0; j < R; ++j) {
      if ((j * kBlk + (t & ~63)) >= n) break;
      xr[j] += alpha * s_p[j * kBlk + t];
      rr[j] -= alpha * s_q[j * kBlk + t];
      rz += rr[j] * (di[j] * rr[j]);
      r2 += rr[j] * rr[j];
    }
    const double2 S = blk_sum2(rz, r2, s_red[1]);
    RR = S.y;
    ++it;
    const bool conv = RR <= stop_rr;
    if (conv || it >= maxiter) {
      done = 1;
      status = conv ? 0 : NGPB_E_NOCONV;
      break;
    }
    const double beta = S.x / rho;
    rho = S.x;
#pragma unroll
    for (int j = 0; j < R; ++j) s_p[j * kBlk + t] = di[j] * rr[j] + beta * s_p[j * kBlk + t];
    __syncthreads();
  }
#pragma unroll
  for (int j = 0; j < R; ++j) {
    const int row = j * kBlk + t;
    if (row < n) {
      x[row] = xr[j];
      r[row] = rr[j];
      p[row] = s_p[row];
    }
  }
  if (t == 0) {
    ks->rho = rho;
    ks->rr = RR;
    ks->iter = it;
    ks->done = done;
    ks->status = status;
  }
}

// runs a system to its end; poll copies *ks to the host and says whether it is done
template <typename Poll>
void run_pcg_block(hipStream_t s, int64_t n, const int32_t* rowptr, const double* val, const SliceRec* recs,
                   const double* dinv, const double* b, double* x, double* r, double* p, KrylovScalars* ks, double tol, int maxiter, Poll poll) {
  const auto k = n <= kBlk ? k_pcg_block<1> : n <= 2 * kBlk ? k_pcg_block<2> : k_pcg_block<4>;
  for (int first = 1;; first = 0) {
    hipLaunchKernelGGL(k, dim3(1), dim3(kBlk), 0, s, (int)n, rowptr, val, recs, dinv, b, x, r, p, ks, tol * tol,
                       maxiter, first, 1024);
    NGPB_HIP(hipGetLastError());
    if (poll()) return;
  }
}

unsigned spmv64_grid(ngpb_ctx* c, bool records) {
  const int64_t need = std::max<int64_t>(1, (c->n + kBS - 1) / kBS);
  if (c->spmv_sched == 0) return (unsigned)std::min<int64_t>(need, 2048);
  int& resident = c->csr_resident[records];
  if (resident <= 0) {
    int cus = 0, per_cu = 0;
    NGPB_HIP(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, c->device));
    if (records) NGPB_HIP(hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, k_spmv64_rec<1>, kBS, 0));
    else NGPB_HIP(hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, (k_spmv64<true, 1>), kBS, 0));
    resident = std::max(8, (std::max(cus, 1) * std::max(per_cu, 1)) / 8 * 8);
  }
  if (need >= resident) return (unsigned)resident;
  return (unsigned)(c->spmv_sched == 1 ? (need + 7) / 8 * 8 : need);
}

// y = A x with the (x, y) partials, from the slice records or (rec null) the CSR
void launch_product(ngpb_ctx* c, unsigned grid, const double* x, double* y, double* part, const void* rec) {
  const SliceRec* R = static_cast<const SliceRec*>(rec);
  if (!R && c->spmv_sched == 1)
    spmv_launch(c, k_spmv64<true, 1>, dim3(grid), dim3(kBS), c->n, c->rowptr.p, c->col.p, c->val.p, x, y, c->ks.p, part);
  else if (!R)
    spmv_launch(c, k_spmv64<true, 0>, dim3(grid), dim3(kBS), c->n, c->rowptr.p, c->col.p, c->val.p, x, y, c->ks.p, part);
  else if (c->spmv_sched == 1)
    spmv_launch(c, k_spmv64_rec<1>, dim3(grid), dim3(kBS), c->n, c->rowptr.p, c->col.p, c->val.p, R, x, y, c->ks.p, part);
  else
    spmv_launch(c, k_spmv64_rec<0>, dim3(grid), dim3(kBS), c->n, c->rowptr.p, c->col.p, c->val.p, R, x, y, c->ks.p, part);
}

// x = 0, r = b, p = D^-1 b; per block (r, D^-1 r), (b, b)
__global__ void __launch_bounds__(kBS) k_pcg_init(int64_t n, const double* __restrict__ b, const double* __restrict__ dinv,
                                                  double* __restrict__ x, double* __restrict__ r, double* __restrict__ p,
                                                  double* __restrict__ partials) {
  __shared__ double s_red[kBS / 64];
  double rz = 0.0, bb = 0.0;
  for (int64_t i = (int64_t)blockIdx.x * kBS + threadIdx.x; i < n; i += (int64_t)gridDim.x * kBS) {
    const double bi = b[i], zi = dinv[i] * bi;
    x[i] = 0.0;
    r[i] = bi;
    p[i] = zi;
    rz += bi * zi;
    bb += bi * bi;
  }
  rz = dev::block_sum<kBS>(rz, s_red);
  bb = dev::block_sum<kBS>(bb, s_red);
  if (threadIdx.x == 0) {
    partials[2 * blockIdx.x] = rz;
    partials[2 * blockIdx.x + 1] = bb;
  }
}

__global__ void __launch_bounds__(kFin) k_fin_init(KrylovScalars* ks, const double* __restrict__ partials, int np,
                                                   double tol2, int maxiter) {
  __shared__ double s_red[kFin / 64];
  const double RZ = dev::sum_partials<kFin>(partials, np, 2, s_red);
  const double BB = dev::sum_partials<kFin>(partials + 1, np, 2, s_red);
  if (threadIdx.x == 0) {
    ks->rho = RZ;
    ks->rho2[0] = RZ;
    ks->iter2[0] = 0;
    ks->bb = BB;
    ks->rr = BB;
    ks->stop_rr = tol2 * BB;
    ks->iter = 0;
    ks->maxiter = maxiter;
    ks->status = 0;
    ks->done = ks->halt2[0] = ks->halt2[1] = (BB == 0.0) ? 1 : 0;
  }
}

// Iteration of parity par. Every block forms (p, q) from the SpMV partials in the
// same fixed order, so all blocks use the same alpha = rho / (p, q).
// r -= alpha q; per block (r, D^-1 r), (r, r); with X x += alpha p
template <bool X>
__global__ void __launch_bounds__(kBS) k_pcg_update(int64_t n, const double* __restrict__ dinv, double* __restrict__ x,
                                                    double* __restrict__ r, const double* __restrict__ p,
                                                    const double* __restrict__ q, KrylovScalars* ks,
                                                    const double* __restrict__ pq_part, int npq,
                                                    double* __restrict__ partials, int par) {
  __shared__ double s_red[kBS / 64];
  if (ks->done) return;
  const double pq = dev::sum_partials<kBS>(pq_part, npq, 1, s_red);
  const double alpha = ks->rho2[par] / pq;
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    ks->pq = pq;
    ks->alpha2[par] = alpha;
  }
  double rz = 0.0, rr = 0.0;
  for (int64_t i = (int64_t)blockIdx.x * kBS + threadIdx.x; i < n; i += (int64_t)gridDim.x * kBS) {
    if (X) x[i] += alpha * p[i];
    const double ri = r[i] - alpha * q[i];
    r[i] = ri;
    rz += ri * (dinv[i] * ri);
    rr += ri * ri;
  }
  rz = dev::block_sum<kBS>(rz, s_red);
  rr = dev::block_sum<kBS>(rr, s_red);
  if (threadIdx.x == 0) {
    partials[2 * blockIdx.x] = rz;
    partials[2 * blockIdx.x + 1] = rr;
  }
}

// With X x += alpha p; the stop test on ||r||^2 (every block decides alike), then
// beta = (r', z') / (r, z) and p = D^-1 r + beta p. Block 0 records the scalars for the
// next iteration and the host. The last step may be added by the launch that raises the
// stop flag, so a block must not return on a flag that this same launch writes: it tests
// halt2[par], which the launch before has written.
template <bool X>
__global__ void __launch_bounds__(kBS) k_pcg_dir(int64_t n, const double* __restrict__ dinv, double* __restrict__ x,
                                                 const double* __restrict__ r, double* __restrict__ p, KrylovScalars* ks,
                                                 const double* __restrict__ part, int np, int par) {
  __shared__ double s_red[kBS / 64];
  if (!X && ks->done) return;  // nothing is left to do on a stop
  if (X && ks->halt2[par]) {
    if (blockIdx.x == 0 && threadIdx.x == 0) ks->halt2[par ^ 1] = 1;
    return;
  }
  const double RZ = dev::sum_partials<kBS>(part, np, 2, s_red);
  const double RR = dev::sum_partials<kBS>(part + 1, np, 2, s_red);
  const int it = ks->iter2[par] + 1;
  const bool conv = RR <= ks->stop_rr;
  const bool stop = conv || it >= ks->maxiter;
  const double rho = ks->rho2[par];
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    ks->rr = RR;
    ks->iter = it;
    ks->iter2[par ^ 1] = it;
    if (stop) {
      ks->done = 1;
      ks->halt2[par ^ 1] = 1;
      ks->status = conv ? 0 : NGPB_E_NOCONV;
      ks->stop_par = par;
    } else {
      ks->beta = RZ / rho;
      ks->rho = RZ;
      ks->rho2[par ^ 1] = RZ;
    }
  }
  if (!X && stop) return;
  const double alpha = ks->alpha2[par], beta = RZ / rho;
  for (int64_t i = (int64_t)blockIdx.x * kBS + threadIdx.x; i < n; i += (int64_t)gridDim.x * kBS) {
    const double pi = p[i];
    if (X) x[i] += alpha * pi;
    if (!stop) p[i] = dinv[i] * r[i] + beta * pi;
  }
}

// The vector kernels of an iteration. Above kFuseRows bytes count, and x is added to
// where p is read for its own update (k_pcg_dir: 80 bytes per row for both against 88).
// Up to there, latency does, and the store of x hides behind the sums of k_pcg_update. Per
// iteration, x in k_pcg_update and in k_pcg_dir: 8,000 rows 12.0 and 12.3 us, 27,000 12.7
// and 13.0, 91,125 14.1 and 14.3, 421,875 28.0 and 28.1, 1 million 36.7 and 35.4; the two
// kernels alone at 4 million 70.4 and 64.8.
constexpr int64_t kFuseRows = int64_t(1) << 19;
void launch_pcg_vectors(hipStream_t s, unsigned gv, int64_t n, const double* dinv, double* x, double* r, double* p,
                        const double* q, KrylovScalars* ks, const double* pq_part, int npq, double* part, int par) {
  const bool fuse = n > kFuseRows;
  hipLaunchKernelGGL(fuse ? k_pcg_update<false> : k_pcg_update<true>, dim3(gv), dim3(kBS), 0, s, n, dinv, x, r, p, q, ks,
                     pq_part, npq, part, par);
  hipLaunchKernelGGL(fuse ? k_pcg_dir<true> : k_pcg_dir<false>, dim3(gv), dim3(kBS), 0, s, n, dinv, x, r, p, ks, part,
                     (int)gv, par);
}

// update (r, q, dinv read; r written) and direction (dinv, r, p read; p written), and x and
// once or twice p for x += alpha p
double pcg_vector_bytes(int64_t n) { return (double)n * 8.0 * (n > kFuseRows ? 10.0 : 11.0); }

__global__ void k_diag_inv(int64_t n, const int32_t* __restrict__ rowptr, const int32_t* __restrict__ col,
                           const double* __restrict__ val, double* __restrict__ dinv, int* __restrict__ bad) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  double d = 0.0;
  for (int64_t k = rowptr[i]; k < rowptr[i + 1]; ++k) {
    const double v = val[k];
    if (!isfinite(v)) atomicOr(bad, 2);
    if (col[k] == i) d = v;
  }
  if (!(d > 0.0)) atomicOr(bad, 1);
  dinv[i] = 1.0 / d;
}

__global__ void __launch_bounds__(kBS) k_copy(int64_t n16, const uint4* __restrict__ a, uint4* __restrict__ b) {
  for (int64_t i = (int64_t)blockIdx.x * kBS + threadIdx.x; i < n16; i += (int64_t)gridDim.x * kBS) b[i] = a[i];
}

}  // namespace

unsigned vec_grid(int64_t n) {
  return (unsigned)std::max<int64_t>(1, std::min<int64_t>((n + 4 * kBS - 1) / (4 * kBS), 2048));
}

// opens the timing of one SpMV when profiling is on and tag is kProfEvery / 2 modulo
// kProfEvery (tag < 0: always). The solvers poll the host every check_every launches
// (32 by default, a multiple of kProfEvery), so the sample leaves out the first launch
// after each poll, which starts on an idle GPU.
void prof_begin(ngpb_ctx* c, int kind, int64_t tag) {
  c->prof_kind = -1;
  if (!c->profile || (tag >= 0 && tag % kProfEvery != kProfEvery / 2)) return;
  c->prof_kind = kind;
  c->prof_tag = tag;
  c->prof_first = true;
}

void prof_end(ngpb_ctx* c, int kind) {
  (void)kind;
  c->prof_kind = -1;
}

// the event pair for the next kernel of the SpMV being timed
hipEvent_t* prof_pair(ngpb_ctx* c) {
  if (c->prof_kind < 0) return nullptr;
  auto& p = c->kprof[c->prof_kind];
  while (p.ev.size() < p.used + 2) {
    hipEvent_t e;
    NGPB_HIP(hipEventCreate(&e));
    p.ev.push_back(e);
  }
  const size_t k = p.used / 2;
  if (p.tag.size() <= k) {
    p.tag.resize(k + 1);
    p.opens.resize(k + 1);
  }
  p.tag[k] = c->prof_tag;
  p.opens[k] = c->prof_first ? 1 : 0;
  c->prof_first = false;
  hipEvent_t* e = &p.ev[p.used];
  p.used += 2;
  return e;
}

// Call after the stream has been synchronized: adds the timed SpMVs whose tag is below
// `limit` (launches queued after the stop flag exit at once and would bias the
// average; limit < 0 keeps all) and clears the record. An SpMV's time is the sum of
// its kernels' own times.
void prof_collect(ngpb_ctx* c, int kind, int64_t limit) {
  auto& p = c->kprof[kind];
  for (size_t i = 0; i + 1 < p.used; i += 2) {
    if (limit >= 0 && p.tag[i / 2] >= limit) continue;
    float ms = 0.f;
    NGPB_HIP(hipEventElapsedTime(&ms, p.ev[i], p.ev[i + 1]));
    p.ms += ms;
    if (p.opens[i / 2]) ++p.launches;
  }
  p.used = 0;
}

// plain device copy of `bytes` (multiple of 16): reads and writes `bytes` each launch
double time_copy(ngpb_ctx* c, int64_t bytes, int reps) {
  const int64_t n16 = bytes / 16;
  DBuf<uint4> a, b;
  a.resize((size_t)n16);
  b.resize((size_t)n16);
  NGPB_HIP(hipMemsetAsync(a.p, 0, n16 * 16, c->stream));
  const unsigned g = (unsigned)std::min<int64_t>((n16 + kBS - 1) / kBS, 8192);
  hipEvent_t e0, e1;
  NGPB_HIP(hipEventCreate(&e0));
  NGPB_HIP(hipEventCreate(&e1));
  hipLaunchKernelGGL(k_copy, dim3(g), dim3(kBS), 0, c->stream, n16, a.p, b.p);
  NGPB_HIP(hipEventRecord(e0, c->stream));
  for (int i = 0; i < reps; ++i) hipLaunchKernelGGL(k_copy, dim3(g), dim3(kBS), 0, c->stream, n16, a.p, b.p);
  NGPB_HIP(hipEventRecord(e1, c->stream));
  NGPB_HIP(hipEventSynchronize(e1));
  NGPB_HIP(hipGetLastError());
  float ms = 0.f;
  NGPB_HIP(hipEventElapsedTime(&ms, e0, e1));
  (void)hipEventDestroy(e0);
  (void)hipEventDestroy(e1);
  return (double)ms / std::max(reps, 1);
}

void ensure_reduce(ngpb_ctx* c, int64_t blocks) {
  const size_t need = (size_t)std::max<int64_t>(blocks, 2048) * 4;
  if (c->red.partials.n < need) c->red.partials.resize(need);
  if (!c->ks.p) c->ks.resize(1);
  if (!c->ks_host) NGPB_HIP(hipHostMalloc((void**)&c->ks_host, sizeof(KrylovScalars), hipHostMallocDefault));
}

namespace {
// 1 / diagonal, its checks and, if asked for, the slice records with the counts of slices
// without one and of diagonals
void check_operator_records(ngpb_ctx* c, bool records, int* staged = nullptr, int* diags = nullptr) {
  c->dinv.resize((size_t)c->n);
  DBuf<int> bad;
  bad.resize(3);
  NGPB_HIP(hipMemsetAsync(bad.p, 0, 3 * sizeof(int), c->stream));
  hipLaunchKernelGGL(k_diag_inv, dim3(blocks_for(c->n, 256)), dim3(256), 0, c->stream, c->n, c->rowptr.p, c->col.p,
                     c->val.p, c->dinv.p, bad.p);
  if (records) {
    const int64_t ns = (c->n + 63) / 64;
    c->slice_rec.reserve((size_t)ns * sizeof(SliceRec));
    hipLaunchKernelGGL(k_slice_rec, dim3(blocks_for(ns, kBS / 64)), dim3(kBS), 0, c->stream, c->n, c->rowptr.p,
                       c->col.p, c->val.p, reinterpret_cast<SliceRec*>(c->slice_rec.p), bad.p);
  }
  NGPB_HIP(hipGetLastError());
  int hb[3] = {0, 0, 0};
  NGPB_HIP(hipMemcpyAsync(hb, bad.p, sizeof(hb), hipMemcpyDeviceToHost, c->stream));
  NGPB_HIP(hipStreamSynchronize(c->stream));
  NGPB_REQUIRE(!(hb[0] & 2), NGPB_E_NUMERIC, "operator holds NaN or Inf entries");
  NGPB_REQUIRE(!(hb[0] & 1), NGPB_E_NUMERIC, "operator has a zero or negative diagonal entry");
  if (staged) *staged = hb[1];
  if (diags) *diags = hb[2];
}
}  // namespace

void spmv_fp64_dot(ngpb_ctx* c, const double* x, double* y, double* partials, const void* rec) {
  launch_product(c, spmv64_grid(c, rec != nullptr), x, y, partials, rec);
}

unsigned spmv_fp64_grid(ngpb_ctx* c, const void* rec) { return spmv64_grid(c, rec != nullptr); }

double spmv_fp64_bytes(const ngpb_ctx* c) {
  // nnz (value + column) + row pointers + x read + y written
  return (double)c->nnz * (8.0 + 4.0) + (double)(c->n + 1) * 4.0 + (double)c->n * 16.0;
}

void spmv_fp64(ngpb_ctx* c, const double* x, double* y) {
  const unsigned grid = spmv64_grid(c, false);
  const KrylovScalars* ks = nullptr;
  double* part = nullptr;
  if (c->spmv_sched == 1)
    spmv_launch(c, k_spmv64<false, 1>, dim3(grid), dim3(kBS), c->n, c->rowptr.p, c->col.p, c->val.p, x, y, ks, part);
  else
    spmv_launch(c, k_spmv64<false, 0>, dim3(grid), dim3(kBS), c->n, c->rowptr.p, c->col.p, c->val.p, x, y, ks, part);
  NGPB_HIP(hipGetLastError());
}

double time_spmv_fp64(ngpb_ctx* c, int reps) {
  c->p.reserve((size_t)c->n);
  c->q.reserve((size_t)c->n);
  NGPB_HIP(hipMemsetAsync(c->p.p, 0, c->n * sizeof(double), c->stream));
  hipEvent_t e0, e1;
  NGPB_HIP(hipEventCreate(&e0));
  NGPB_HIP(hipEventCreate(&e1));
  spmv_fp64(c, c->p.p, c->q.p);  // warm-up
  NGPB_HIP(hipEventRecord(e0, c->stream));
  for (int i = 0; i < reps; ++i) spmv_fp64(c, c->p.p, c->q.p);
  NGPB_HIP(hipEventRecord(e1, c->stream));
  NGPB_HIP(hipEventSynchronize(e1));
  float ms = 0.f;
  NGPB_HIP(hipEventElapsedTime(&ms, e0, e1));
  (void)hipEventDestroy(e0);
  (void)hipEventDestroy(e1);
  return (double)ms / std::max(reps, 1);
}

void check_operator(ngpb_ctx* c) { check_operator_records(c, false); }

const void* slice_records(ngpb_ctx* c, bool* block) {
  int staged = 0, diags = 0;
  check_operator_records(c, true, &staged, &diags);
  if (block) *block = use_block(c->n, staged, diags);
  return use_records(c->n, staged) ? c->slice_rec.p : nullptr;
}

namespace {
// A solve in one block launches no product of its own to time: profiling times as many
// single ones after it, so that it changes no result.
void time_products(ngpb_ctx* c, unsigned grid, double* part, const void* rec) {
  KrylovScalars& h = *c->ks_host;
  const int done = h.done;
  h.done = 0;
  NGPB_HIP(hipMemcpyAsync(c->ks.p, &h, sizeof(h), hipMemcpyHostToDevice, c->stream));
  for (int64_t k = kProfEvery / 2; k < h.iter; k += kProfEvery) {
    prof_begin(c, 0, k);
    launch_product(c, grid, c->p.p, c->q.p, part, rec);
    prof_end(c, 0);
  }
  NGPB_HIP(hipGetLastError());
  NGPB_HIP(hipStreamSynchronize(c->stream));
  h.done = done;
  prof_collect(c, 0, h.iter);
}
}  // namespace

void solve_fp64(ngpb_ctx* c, const ngpb_solve_opts& o, ngpb_solve_stats& st) {
  const int64_t n = c->n;
  bool block = false;
  const void* rec = slice_records(c, &block);
  c->x.resize((size_t)n);
  c->r.resize((size_t)n);
  c->p.reserve((size_t)n);
  c->q.reserve((size_t)n);
  const unsigned gs = spmv64_grid(c, rec != nullptr), gv = vec_grid(n);
  ensure_reduce(c, std::max<int64_t>(gs, 2048) + 2 * (int64_t)gv);
  double* part = c->red.partials.p;
  KrylovScalars* ks = c->ks.p;
  hipEvent_t e0, e1;
  NGPB_HIP(hipEventCreate(&e0));
  NGPB_HIP(hipEventCreate(&e1));
  NGPB_HIP(hipEventRecord(e0, c->stream));
  const auto poll = [&]() {
    NGPB_HIP(hipMemcpyAsync(c->ks_host, ks, sizeof(KrylovScalars), hipMemcpyDeviceToHost, c->stream));
    NGPB_HIP(hipStreamSynchronize(c->stream));
    return c->ks_host->done != 0;
  };
  if (block) {
    run_pcg_block(c->stream, n, c->rowptr.p, c->val.p, static_cast<const SliceRec*>(rec), c->dinv.p, c->rhs.p,
                  c->x.p, c->r.p, c->p.p, ks, o.tol, o.maxiter, poll);
  } else {
    hipLaunchKernelGGL(k_pcg_init, dim3(gv), dim3(kBS), 0, c->stream, n, c->rhs.p, c->dinv.p, c->x.p, c->r.p, c->p.p, part);
    hipLaunchKernelGGL(k_fin_init, dim3(1), dim3(kFin), 0, c->stream, ks, part, (int)gv, o.tol * o.tol, o.maxiter);
    NGPB_HIP(hipGetLastError());
    // partial-sum regions: SpMV (p, q) and update (r, z), (r, r)
    double* ppq = part;
    double* pup = part + std::max<int64_t>(gs, 2048);
    const int chunk = std::max(1, o.check_every);
    for (int64_t launch = 0;;) {
      for (int k = 0; k < chunk; ++k, ++launch) {
        const int par = (int)(launch & 1);
        prof_begin(c, 0, launch);
        launch_product(c, gs, c->p.p, c->q.p, ppq, rec);
        prof_end(c, 0);
        launch_pcg_vectors(c->stream, gv, n, c->dinv.p, c->x.p, c->r.p, c->p.p, c->q.p, ks, ppq, (int)gs, pup, par);
      }
      NGPB_HIP(hipGetLastError());
      const bool done = poll();
      prof_collect(c, 0, c->ks_host->iter);
      if (done) break;
    }
  }
  NGPB_HIP(hipEventRecord(e1, c->stream));
  NGPB_HIP(hipEventSynchronize(e1));
  float ms = 0.f;
  NGPB_HIP(hipEventElapsedTime(&ms, e0, e1));
  (void)hipEventDestroy(e0);
  (void)hipEventDestroy(e1);
  if (block && c->profile) time_products(c, gs, part, rec);
  const KrylovScalars& h = *c->ks_host;
  st.status = h.status;
  st.iterations = h.iter;
  st.replacements = 0;
  st.relres = h.bb > 0 ? std::sqrt(h.rr / h.bb) : 0.0;
  st.ms_solve = ms;
  st.bytes_per_iter = spmv_fp64_bytes(c) + pcg_vector_bytes(n);
  c->have_phi = true;
  c->phi_len = c->n;
}

// ------------------------------------------------------------ allocation-free entry point
// ngpb_solve_csr_noalloc runs the CG-Jacobi above on a CSR system the caller keeps in
// device memory, with its work vectors, partial sums, scalars, flags and slice records in one
// file-scope device array: the call allocates nothing (no hipMalloc / hipFree, no
// pinned host memory, no events), for callers that cannot allocate. Each GPU holds
// its own copy of the array until the process ends; its address on a device is taken
// once with hipGetSymbolAddress, and only that address is handed to kernels and
// copies. Every call on one GPU uses the same array, so calls that overlap on one GPU
// (from several host threads or streams) race; each call initializes what it reads.
constexpr int64_t kNoAllocMaxRows = int64_t(1) << 20;  // 1,048,576 rows
constexpr int64_t kNoAllocPartials = 8192;             // >= 2048 + 2 * 2048
constexpr int64_t kNoAllocRecs = (kNoAllocMaxRows / 64) * (int64_t)(sizeof(SliceRec) / 8);  // in doubles
constexpr int64_t kNoAllocDoubles = 4 * kNoAllocMaxRows + kNoAllocPartials + 64 + kNoAllocRecs;
static __device__ __align__(256) double scratch[kNoAllocDoubles];

namespace {

constexpr int kMaxDevices = 64;
std::mutex g_scratch_mu;
double* g_scratch_ptr[kMaxDevices] = {};

__global__ void k_clear_flags(int* p) { p[threadIdx.x] = 0; }

// Structure of a CSR the library did not build: row pointers from 0 to nnz, non-
// decreasing, columns in [0, n). Sets bit 4 of *bad otherwise; reads col only below nnz.
__global__ void k_csr_check(int64_t n, int64_t nnz, const int32_t* __restrict__ rowptr,
                            const int32_t* __restrict__ col, int* __restrict__ bad) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const int64_t a = rowptr[i], e = rowptr[i + 1];
  if ((i == 0 && a != 0) || (i == n - 1 && e != nnz) || a < 0 || e < a || e > nnz) {
    atomicOr(bad, 4);
    return;
  }
  for (int64_t k = a; k < e; ++k)
    if (col[k] < 0 || col[k] >= n) {
      atomicOr(bad, 4);
      return;
    }
}

// device address of `scratch` on the current device (taken on the first call there)
double* scratch_on(int device) {
  std::lock_guard<std::mutex> lk(g_scratch_mu);
  if (!g_scratch_ptr[device]) {
    void* ptr = nullptr;
    NGPB_HIP(hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch)));
    NGPB_REQUIRE(ptr != nullptr, NGPB_E_HIP, "no device address for the scratch array");
    g_scratch_ptr[device] = static_cast<double*>(ptr);
  }
  return g_scratch_ptr[device];
}

}  // namespace

int64_t noalloc_max_rows() { return kNoAllocMaxRows; }

void solve_csr_noalloc(int device, hipStream_t s, int64_t n, int64_t nnz, const int32_t* rowptr, const int32_t* col,
                       const double* val, const double* b, double* x, double tol, int maxiter, int check_every,
                       ngpb_solve_stats& st) {
  NGPB_REQUIRE(n > 0 && n <= kNoAllocMaxRows, NGPB_E_ARG,
               "ngpb_solve_csr_noalloc takes 1 to 1,048,576 rows (its scratch array is sized for that)");
  double* base = scratch_on(device);
  double* dinv = base;
  double* r = base + kNoAllocMaxRows;
  double* p = base + 2 * kNoAllocMaxRows;
  double* q = base + 3 * kNoAllocMaxRows;
  double* part = base + 4 * kNoAllocMaxRows;
  KrylovScalars* ks = reinterpret_cast<KrylovScalars*>(part + kNoAllocPartials);
  int* bad = reinterpret_cast<int*>(ks + 1);
  SliceRec* recs = reinterpret_cast<SliceRec*>(part + kNoAllocPartials + 64);
  static_assert(sizeof(KrylovScalars) + 3 * sizeof(int) <= 64 * sizeof(double), "scalar area too small");
  const auto t0 = std::chrono::steady_clock::now();
  hipLaunchKernelGGL(k_clear_flags, dim3(1), dim3(3), 0, s, bad);
  hipLaunchKernelGGL(k_csr_check, dim3(blocks_for(n, 256)), dim3(256), 0, s, n, nnz, rowptr, col, bad);
  NGPB_HIP(hipGetLastError());
  int hb[3] = {0, 0, 0};
  NGPB_HIP(hipMemcpyAsync(hb, bad, sizeof(hb), hipMemcpyDeviceToHost, s));
  NGPB_HIP(hipStreamSynchronize(s));
  NGPB_REQUIRE(!(hb[0] & 4), NGPB_E_ARG, "row pointers must run from 0 to nnz without decreasing, columns in [0, n)");
  hipLaunchKernelGGL(k_diag_inv, dim3(blocks_for(n, 256)), dim3(256), 0, s, n, rowptr, col, val, dinv, bad);
  hipLaunchKernelGGL(k_slice_rec, dim3(blocks_for((n + 63) / 64, kBS / 64)), dim3(kBS), 0, s, n, rowptr, col, val, recs,
                     bad);
  NGPB_HIP(hipGetLastError());
  NGPB_HIP(hipMemcpyAsync(hb, bad, sizeof(hb), hipMemcpyDeviceToHost, s));
  NGPB_HIP(hipStreamSynchronize(s));
  NGPB_REQUIRE(!(hb[0] & 2), NGPB_E_NUMERIC, "operator holds NaN or Inf entries");
  NGPB_REQUIRE(!(hb[0] & 1), NGPB_E_NUMERIC, "operator has a zero or negative diagonal entry");
  KrylovScalars h;
  std::memset(&h, 0, sizeof(h));
  const auto poll = [&]() {
    NGPB_HIP(hipMemcpyAsync(&h, ks, sizeof(KrylovScalars), hipMemcpyDeviceToHost, s));
    NGPB_HIP(hipStreamSynchronize(s));
    return h.done != 0;
  };
  if (use_block(n, hb[1], hb[2])) {
    run_pcg_block(s, n, rowptr, val, recs, dinv, b, x, r, p, ks, tol, maxiter, poll);
  } else {
    // the launch shapes of ngpb_solve under SpMV schedule 0
    const unsigned gs = (unsigned)std::min<int64_t>(std::max<int64_t>(1, (n + kBS - 1) / kBS), 2048);
    const unsigned gv = vec_grid(n);
    double* ppq = part;
    double* pup = part + 2048;
    hipLaunchKernelGGL(k_pcg_init, dim3(gv), dim3(kBS), 0, s, n, b, dinv, x, r, p, pup);
    hipLaunchKernelGGL(k_fin_init, dim3(1), dim3(kFin), 0, s, ks, pup, (int)gv, tol * tol, maxiter);
    NGPB_HIP(hipGetLastError());
    const bool records = use_records(n, hb[1]);
    const int chunk = std::max(1, check_every);
    for (int64_t launch = 0;;) {
      for (int k = 0; k < chunk; ++k, ++launch) {
        const int par = (int)(launch & 1);
        if (records)
          hipLaunchKernelGGL(k_spmv64_rec<0>, dim3(gs), dim3(kBS), 0, s, n, rowptr, col, val, recs, p, q, ks, ppq);
        else
          hipLaunchKernelGGL((k_spmv64<true, 0>), dim3(gs), dim3(kBS), 0, s, n, rowptr, col, val, p, q, ks, ppq);
        launch_pcg_vectors(s, gv, n, dinv, x, r, p, q, ks, ppq, (int)gs, pup, par);
      }
      NGPB_HIP(hipGetLastError());
      if (poll()) break;
    }
  }
  st.status = h.status;
  st.iterations = h.iter;
  st.replacements = 0;
  st.relres = h.bb > 0 ? std::sqrt(h.rr / h.bb) : 0.0;
  st.ms_solve = std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now() - t0).count();
  // SpMV (12 nnz + 4 (n + 1) + 16 n) + update and direction vector streams, as ngpb_solve
  st.bytes_per_iter = 12.0 * (double)nnz + 4.0 * (double)(n + 1) + 16.0 * (double)n + pcg_vector_bytes(n);
}

}  // namespace ngpb
