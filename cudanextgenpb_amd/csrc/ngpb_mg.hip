// Geometric multigrid preconditioner of the mixed-precision solve.
//
// Why. The FP32 inner CG with Jacobi scaling needs 300-900 iterations, a number that
// grows with the grid. On an octree mesh the coarse problems are cheap: uniform grids of
// twice, four times ... the finest spacing with seven-point operators, whose memory is
// an eighth of the finest grid's and whose kernels stream contiguous arrays. A V(1,1)
// cycle as CG's preconditioner takes 20-30 iterations on every size, each three compact
// SpMVs instead of one.
//
// Levels. Level 0 is the octree operator itself (compact FP32 form, unit diagonal after
// the symmetric Jacobi scaling, smoothed by one damped Jacobi step before and after the
// coarse correction). Level l >= 1 is the uniform grid of spacing 2^l hf over the mesh's
// box, with zero values on the box faces; where the cell count of a level is odd, the
// next level's last cell reaches past the box. Its edge coefficients come from the
// leaves' edge conductances: per cell and axis the harmonic mean along the axis of the
// arithmetic means across it, the screening term the mean of the cell's corners.
//
// Transfers. Nodes with a leaf of edge hf or 2 hf around them are copied into a dense
// array of the finest grid (zero where the octree has no node) and restricted from
// there by full weighting; their correction is the trilinear interpolation of level 1.
// A node whose leaves all have edges of at least 2^l hf, l >= 2, lies on grid l and
// exchanges its residual and correction with that level directly. Restriction is the
// transpose of prolongation and the smoothers are symmetric, so the cycle is a symmetric
// positive definite operator and plain CG applies.
//
// Measured (tolerance 1e-10, solve alone, against Jacobi scaling): 8.04M unknowns 556 ->
// 29 iterations, 57.8 -> 14.9 ms; 63.3M unknowns 892 iterations, 656 ms -> whole step 801
// -> 283 ms; 274,625 unknowns (64^3 cells) 340 -> 22, 5.9 -> 2.1 ms; 47,302 unknowns 223
// -> 26, 4.2 -> 2.6 ms. A cycle streams from HBM at the large sizes and is bound by the
// latency of its ~20 launches at the small ones.
//
// All reductions have a fixed order and no kernel uses atomics on values: a repeated
// solve is bit-identical.
#include <algorithm>
#include <cmath>
#include <cstring>
#include <vector>

#include "ngpb_internal.h"
#include "ngpb_mg_dev.h"

namespace ngpb {
MeshView mesh_view_of(const ngpb_ctx* c);

namespace {

constexpr int kBS = 256;

// ------------------------------------------------------------------ setup
__device__ __forceinline__ int axis_index(double x, double x0, double inv_h, int* bad) {
  const double u = (x - x0) * inv_h;
  const double r = rint(u);
  if (fabs(u - r) > 1e-5 || r < 0.0 || r > 1022.0) {
    *bad = 1;
    return 0;
  }
  return (int)r;
}

// Per-block minimum of the leaf edges and minimum / maximum node coordinates; leaves
// must be cubes. out: 7 per block (edge, min xyz, max xyz).
__global__ void __launch_bounds__(kBS) k_mg_extent(MeshView m, double* __restrict__ out, int* __restrict__ bad) {
  __shared__ double s[7][kBS];
  double e = INFINITY, lo[3] = {INFINITY, INFINITY, INFINITY}, hi[3] = {-INFINITY, -INFINITY, -INFINITY};
  for (int64_t l = (int64_t)blockIdx.x * kBS + threadIdx.x; l < m.L; l += (int64_t)gridDim.x * kBS) {
    const int32_t c0 = m.leaf_corner[8 * l], c7 = m.leaf_corner[8 * l + 7];
    const double h = dev::corner_coord(m, c7, 0) - dev::corner_coord(m, c0, 0);
    for (int d = 1; d < 3; ++d)
      if (!(fabs(dev::corner_coord(m, c7, d) - dev::corner_coord(m, c0, d) - h) <= 1e-6 * h)) *bad = 1;
    e = fmin(e, h);
  }
  for (int64_t i = (int64_t)blockIdx.x * kBS + threadIdx.x; i < m.N; i += (int64_t)gridDim.x * kBS)
    for (int d = 0; d < 3; ++d) {
      const double v = m.node_xyz[3 * i + d];
      lo[d] = fmin(lo[d], v);
      hi[d] = fmax(hi[d], v);
    }
  s[0][threadIdx.x] = e;
  for (int d = 0; d < 3; ++d) {
    s[1 + d][threadIdx.x] = lo[d];
    s[4 + d][threadIdx.x] = hi[d];
  }
  __syncthreads();
  for (int w = kBS / 2; w > 0; w >>= 1) {
    if ((int)threadIdx.x < w)
      for (int k = 0; k < 7; ++k) {
        const double a = s[k][threadIdx.x], b = s[k][threadIdx.x + w];
        s[k][threadIdx.x] = k < 4 ? fmin(a, b) : fmax(a, b);
      }
    __syncthreads();
  }
  if (threadIdx.x < 7) out[7 * blockIdx.x + threadIdx.x] = s[threadIdx.x][0];
}

// Leaf levels, and the leaf id at each leaf's anchor cell of the finest grid.
__global__ void __launch_bounds__(kBS) k_mg_leaf_map(MeshView m, MgBox g, int32_t* __restrict__ map,
                                                     uint8_t* __restrict__ level, int* __restrict__ bad) {
  const int64_t l = (int64_t)blockIdx.x * kBS + threadIdx.x;
  if (l >= m.L) return;
  const int32_t c0 = m.leaf_corner[8 * l], c7 = m.leaf_corner[8 * l + 7];
  int a[3], b[3];
  int wrong = 0;
  for (int d = 0; d < 3; ++d) {
    a[d] = axis_index(dev::corner_coord(m, c0, d), g.x0[d], g.inv_h, &wrong);
    b[d] = axis_index(dev::corner_coord(m, c7, d), g.x0[d], g.inv_h, &wrong);
  }
  const int e = b[0] - a[0];
  const int s = 31 - __clz(max(e, 1));
  if (wrong || e != (1 << s) || s > 10 || ((a[0] | a[1] | a[2]) & (e - 1)) || a[0] >= g.n[0] || a[1] >= g.n[1] ||
      a[2] >= g.n[2]) {
    *bad = 1;
    return;
  }
  level[l] = (uint8_t)s;
  map[((int64_t)a[2] * g.n[1] + a[1]) * g.n[0] + a[0]] = (int32_t)l;
}

// node level: the smallest level among its leaves; one launch per level, coarse first,
// so that the finest leaf's value stays (all writers of a launch write the same value)
__global__ void __launch_bounds__(kBS) k_mg_node_level(int64_t L, const int32_t* __restrict__ corner,
                                                       const uint8_t* __restrict__ level, int lo, int hi,
                                                       uint8_t* __restrict__ nlev) {
  const int64_t l = (int64_t)blockIdx.x * kBS + threadIdx.x;
  if (l >= L) return;
  const int s = level[l];
  if (s < lo || s > hi) return;
  for (int i = 0; i < 8; ++i) {
    const int32_t c = corner[8 * l + i];
    if (c >= 0) nlev[c] = (uint8_t)lo;
  }
}

// Packed position of every row (10 bits per axis; 2 bits: 0 through the dense array, d:
// directly on level d + 1) and its transfer scale, the square root of its diagonal (0
// for the decoupled Dirichlet rows). Counts rows for which "on a box face" and
// "decoupled" disagree: the coarse levels hold zeros on the faces and nowhere else.
__global__ void __launch_bounds__(kBS) k_mg_rows(int64_t n, const double* __restrict__ xyz, MgBox g,
                                                 const int32_t* __restrict__ rowptr, const double* __restrict__ dscale,
                                                 const int32_t* __restrict__ perm, const uint8_t* __restrict__ nlev,
                                                 int max_direct, uint32_t* __restrict__ pos, float* __restrict__ sd,
                                                 int* __restrict__ bad) {
  const int64_t r = (int64_t)blockIdx.x * kBS + threadIdx.x;
  if (r >= n) return;
  const int64_t i = perm ? (int64_t)perm[r] : r;
  int wrong = 0, p[3];
  bool face = false;
  for (int d = 0; d < 3; ++d) {
    p[d] = axis_index(xyz[3 * i + d], g.x0[d], g.inv_h, &wrong);
    if (p[d] > g.n[d]) wrong = 1;
    face |= p[d] == 0 || p[d] == g.n[d];
  }
  const bool alone = rowptr[i + 1] - rowptr[i] == 1;
  int direct = nlev[i] >= 2 ? min((int)nlev[i] - 1, max_direct) : 0;
  if (nlev[i] == 255) wrong = 1;
  if (direct && ((p[0] | p[1] | p[2]) & ((2 << direct) - 1))) wrong = 1;
  if (wrong || alone != face) *bad = 1;
  pos[r] = (uint32_t)p[0] | (uint32_t)p[1] << 10 | (uint32_t)p[2] << 20 | (uint32_t)direct << 30;
  sd[r] = alone ? 0.f : (float)(1.0 / dscale[r]);
}

// coefficients of leaf l of edge 1 / inv: per axis the mean of its four edges'
// permittivities, and the mean screening term of its corners
__device__ __forceinline__ float4 leaf_cell(const MeshView& m, int64_t l, double inv, const double* c_edge,
                                            const double* reac) {
  // edge order: x edges 0 2 4 6, y edges 1 3 5 7, z edges 8 .. 11; c_edge = eps h / 4
  const double* c = c_edge + 12 * l;
  double r = 0.0;
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const int32_t k = m.leaf_corner[8 * l + i];
    if (k >= 0) {
      r += reac[k];
    } else {
      const int64_t hh = -1 - (int64_t)k;
      const int np = m.hang_np[hh];
      double t = 0.0;
      for (int j = 0; j < np; ++j) t += reac[m.hang_par[4 * hh + j]];
      r += t / np;
    }
  }
  return make_float4((float)((c[0] + c[2] + c[4] + c[6]) * inv), (float)((c[1] + c[3] + c[5] + c[7]) * inv),
                     (float)((c[8] + c[9] + c[10] + c[11]) * inv), (float)(r * 0.125));
}

__device__ __forceinline__ float hmean(float a, float b) { return 2.f * a * b / (a + b); }

// coefficients of a coarse cell from its eight children (bit0 = x, bit1 = y, bit2 = z):
// harmonic means along the axis of the arithmetic means across it
__device__ __forceinline__ float4 merge_cells(const float4* q) {
  float4 o;
  o.x = hmean(0.25f * (q[0].x + q[2].x + q[4].x + q[6].x), 0.25f * (q[1].x + q[3].x + q[5].x + q[7].x));
  o.y = hmean(0.25f * (q[0].y + q[1].y + q[4].y + q[5].y), 0.25f * (q[2].y + q[3].y + q[6].y + q[7].y));
  o.z = hmean(0.25f * (q[0].z + q[1].z + q[2].z + q[3].z), 0.25f * (q[4].z + q[5].z + q[6].z + q[7].z));
  float s = 0.f;
  for (int i = 0; i < 8; ++i) s += q[i].w;
  o.w = 0.125f * s;
  return o;
}

// Cells of level 1 (edge 2 hf) from the leaves, eight lanes a cell: eight leaves of edge
// hf, one per lane, or the one larger leaf that holds the cell (found at its anchor). One
// thread per cell took 1.0 ms on the 8M-node mesh, 96-byte leaf records read serially.
__global__ void __launch_bounds__(kBS) k_mg_cells1(MeshView m, MgBox g, int cx, int cy, int cz,
                                                   const int32_t* __restrict__ map, const uint8_t* __restrict__ level,
                                                   const double* __restrict__ c_edge,
                                                   const double* __restrict__ reac, float4* __restrict__ cells,
                                                   int* __restrict__ bad) {
  const int64_t t = ((int64_t)blockIdx.x * kBS + threadIdx.x) >> 3;
  const int c = threadIdx.x & 7;
  const bool valid = t < (int64_t)cx * cy * cz;
  float4 q = make_float4(1.f, 1.f, 1.f, 0.f);
  if (valid) {
    const int I = (int)(t % cx), J = (int)(t / cx % cy), K = (int)(t / ((int64_t)cx * cy));
    auto at = [&](int i, int j, int k) { return map[((int64_t)k * g.n[1] + j) * g.n[0] + i]; };
    int32_t l = at(min(2 * I + (c & 1), g.n[0] - 1), min(2 * J + ((c >> 1) & 1), g.n[1] - 1),
                   min(2 * K + (c >> 2), g.n[2] - 1));
    int s = 0;
    if (l < 0 || level[l] != 0) {
      l = -1;
      for (s = 1; s <= 10 && l < 0; ++s) {
        const int k = ~((1 << s) - 1);
        const int32_t cand = at(2 * I & k, 2 * J & k, 2 * K & k);
        if (cand >= 0 && level[cand] >= s) l = cand;
      }
      if (l >= 0) s = level[l];
    }
    if (l < 0) *bad = 1;
    else q = leaf_cell(m, l, g.inv_h / (double)(1 << s), c_edge, reac);
  }
  // harmonic mean along the axis of the arithmetic means across it
  auto axis = [&](float v, int along, int b0, int b1) {
    v += __shfl_xor(v, b0, 64);
    v += __shfl_xor(v, b1, 64);
    return hmean(0.25f * v, 0.25f * __shfl_xor(v, along, 64));
  };
  float4 o;
  o.x = axis(q.x, 1, 2, 4);
  o.y = axis(q.y, 2, 1, 4);
  o.z = axis(q.z, 4, 1, 2);
  o.w = q.w;
  for (int b = 1; b <= 4; b *= 2) o.w += __shfl_xor(o.w, b, 64);
  o.w *= 0.125f;
  if (valid && c == 0) cells[t] = o;
}

__global__ void __launch_bounds__(kBS) k_mg_cells(int fx, int fy, int fz, const float4* __restrict__ f, int cx, int cy,
                                                  int cz, float4* __restrict__ cells) {
  const int64_t t = (int64_t)blockIdx.x * kBS + threadIdx.x;
  if (t >= (int64_t)cx * cy * cz) return;
  const int I = (int)(t % cx), J = (int)(t / cx % cy), K = (int)(t / ((int64_t)cx * cy));
  float4 q[8];
  for (int c = 0; c < 8; ++c)
    q[c] = f[((int64_t)min(2 * K + (c >> 2), fz - 1) * fy + min(2 * J + ((c >> 1) & 1), fy - 1)) * fx +
             min(2 * I + (c & 1), fx - 1)];
  cells[t] = merge_cells(q);
}

// conductances to the +x, +y, +z neighbours and inverse diagonal of every node of a
// level; zero on the faces, and the level's vectors cleared
__global__ void __launch_bounds__(kBS) k_mg_edges(MgGrid g, float h, const float4* __restrict__ cells) {
  const int i = blockIdx.x * 64 + (threadIdx.x & 63), j = blockIdx.y * 4 + (threadIdx.x >> 6), k = blockIdx.z;
  if (i >= g.pitch || j > g.cy) return;
  const int64_t o = g.at(i, j, k);
  g.b[o] = 0.f;
  g.x[o] = 0.f;
  g.t[o] = 0.f;
  if (g.f) g.f[o] = 0.f;
  float ex = 0.f, ey = 0.f, ez = 0.f, d = 0.f;
  if (i <= g.cx) {
    auto cell = [&](int a, int b, int c) {
      return cells[((int64_t)min(max(c, 0), g.cz - 1) * g.cy + min(max(b, 0), g.cy - 1)) * g.cx +
                   min(max(a, 0), g.cx - 1)];
    };
    float sx = 0.f, sy = 0.f, sz = 0.f, sm = 0.f, se = 0.f;
    for (int c = 0; c < 8; ++c) {
      const int a = i - 1 + (c & 1), b = j - 1 + ((c >> 1) & 1), e = k - 1 + (c >> 2);
      const float4 q = cell(a, b, e);
      se += q.x + q.y + q.z;
      sm += q.w;
      if (c & 1) sx += q.x;
      if (c & 2) sy += q.y;
      if (c & 4) sz += q.z;
    }
    ex = 0.25f * h * sx;
    ey = 0.25f * h * sy;
    ez = 0.25f * h * sz;
    if (g.inner(i, j, k)) d = 1.f / (0.25f * h * se + 0.125f * h * h * h * sm);
  }
  g.ex[o] = ex;
  g.ey[o] = ey;
  g.ez[o] = ez;
  g.dinv[o] = d;
}

// ------------------------------------------------------------------ cycle
// The levels' kernels: four nodes of a grid row per thread (mg_*_quad), one thread in a
// flat index per quad.

__global__ void __launch_bounds__(kBS) k_mg_resid(MgGrid g, const KrylovScalars* ks) {
  if (ks->done) return;
  mg_resid_quad(g, blockIdx.x * kBS + threadIdx.x);
}

__global__ void __launch_bounds__(kBS) k_mg_restrict(MgGrid g, const float* __restrict__ t, int pitch, int rows,
                                                     const KrylovScalars* ks) {
  if (ks->done) return;
  mg_restrict_pair(g, t, pitch, rows, blockIdx.x * kBS + threadIdx.x);
}

__global__ void __launch_bounds__(kBS) k_mg_prolong(MgGrid g, MgGrid c, const KrylovScalars* ks) {
  if (ks->done) return;
  mg_prolong_quad(g, c, blockIdx.x * kBS + threadIdx.x);
}

__global__ void __launch_bounds__(kBS) k_mg_smooth(MgGrid g, const KrylovScalars* ks) {
  if (ks->done) return;
  mg_smooth_quad(g, blockIdx.x * kBS + threadIdx.x);
}

__global__ void __launch_bounds__(kMgBottomBS) k_mg_bottom(MgHierarchy h, const KrylovScalars* ks) {
  extern __shared__ float s_mem[];
  if (ks->done) return;
  mg_bottom(h, s_mem);
}

// ------------------------------------------------------------------ octree level
// Stop test on (r, r) of the previous update (every block decides alike), then the
// residual after the first smoothing step, r - omega Ahat r, in unscaled units into the
// dense array or the direct levels' right-hand sides.
__global__ void __launch_bounds__(kBS) k_mgf_embed(MgHierarchy h, int64_t n, const uint32_t* __restrict__ pos,
                                                   const float* __restrict__ sd, const float* __restrict__ r,
                                                   const float* __restrict__ ar, KrylovScalars* ks,
                                                   const double* __restrict__ rr_part, int npr, int par, int first) {
  __shared__ double s_red[kBS / 64];
  if (ks->done) return;
  if (!first) {
    const double RR = dev::sum_partials<kBS>(rr_part, npr, 1, s_red);
    const int it = ks->iter2[par];
    const bool stop = !(RR > ks->stop_rr) || it >= ks->maxiter;  // also on NaN
    if (blockIdx.x == 0 && threadIdx.x == 0) {
      ks->rr = RR;
      ks->iter = it;
      if (stop) {
        ks->done = 1;
        ks->stop_par = par;
      }
    }
    if (stop) return;
  }
  for (int64_t q = (int64_t)blockIdx.x * kBS + threadIdx.x; q < n; q += (int64_t)gridDim.x * kBS)
    mg_embed(h, pos[q], sd[q] * fmaf(-kMgOmega, ar[q], r[q]));
}

// rows a thread has in flight: a row's position leads to its coarse values, a chain of
// two memory latencies (8M rows: 43 us with one row in flight, 38 with four)
constexpr int kUnroll = 4;

// z0 = omega r + scaled coarse correction; per block (z0, r - omega Ahat r), which with
// omega (r, r) makes (r, z) of z = z0 + omega (r - Ahat z0): Ahat is symmetric
__global__ void __launch_bounds__(kBS) k_mgf_correct(MgHierarchy h, int64_t n, const uint32_t* __restrict__ pos,
                                                     const float* __restrict__ sd, const float* __restrict__ r,
                                                     const float* __restrict__ ar, float* __restrict__ z,
                                                     const KrylovScalars* ks, double* __restrict__ part) {
  __shared__ double s_red[kBS / 64];
  if (ks->done) return;
  double s = 0.0;
  const int64_t step = (int64_t)gridDim.x * kBS;
  for (int64_t b = (int64_t)blockIdx.x * kBS; b < n; b += kUnroll * step) {
    uint32_t p[kUnroll];
    float ri[kUnroll], ai[kUnroll], si[kUnroll], e[kUnroll];
#pragma unroll
    for (int u = 0; u < kUnroll; ++u) {
      const int64_t q = min(b + u * step + threadIdx.x, n - 1);
      p[u] = pos[q];
      ri[u] = r[q];
      ai[u] = ar[q];
      si[u] = sd[q];
    }
#pragma unroll
    for (int u = 0; u < kUnroll; ++u) e[u] = mg_correction(h, p[u], b + u * step + threadIdx.x < n);
#pragma unroll
    for (int u = 0; u < kUnroll; ++u) {
      const int64_t q = b + u * step + threadIdx.x;
      if (q < n) {
        const float zi = fmaf(si[u], e[u], kMgOmega * ri[u]);
        z[q] = zi;
        s += (double)zi * (double)fmaf(-kMgOmega, ai[u], ri[u]);
      }
    }
  }
  s = dev::block_sum<kBS>(s, s_red);
  if (threadIdx.x == 0) part[blockIdx.x] = s;
}

// xhat += alpha p of the previous iteration; z = z0 + omega (r - Ahat z0) and
// p = z + beta p, beta = (r, z) / (r, z) of the previous iteration
__global__ void __launch_bounds__(kBS) k_mgf_dir(int64_t n, const float* __restrict__ z, const float* __restrict__ r,
                                                 const float* __restrict__ az, float* __restrict__ p,
                                                 float* __restrict__ x, KrylovScalars* ks,
                                                 const double* __restrict__ part, int np, int par) {
  __shared__ double s_red[kBS / 64];
  if (ks->done) return;
  const double rz = dev::sum_partials<kBS>(part, np, 1, s_red) + (double)kMgOmega * ks->rr;
  const double old = ks->rho2[par];
  const float beta = old > 0.0 ? (float)(rz / old) : 0.f;
  const float alpha = (float)ks->alpha2[par];
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    ks->rho2[par ^ 1] = rz;
    ks->iter2[par ^ 1] = ks->iter2[par] + 1;
  }
  for (int64_t q = (int64_t)blockIdx.x * kBS + threadIdx.x; q < n; q += (int64_t)gridDim.x * kBS) {
    const float pi = p[q];
    // xhat and Ahat z0 are not read again before everything else has passed the caches
    __builtin_nontemporal_store(fmaf(alpha, pi, __builtin_nontemporal_load(&x[q])), &x[q]);
    p[q] = fmaf(beta, pi, fmaf(kMgOmega, r[q] - __builtin_nontemporal_load(&az[q]), z[q]));
  }
}

// alpha = (r, z) / (p, Ahat p); r -= alpha Ahat p; per block (r, r)
__global__ void __launch_bounds__(kBS) k_mgf_update(int64_t n, float* __restrict__ r, const float* __restrict__ ap,
                                                    KrylovScalars* ks, const double* __restrict__ pq_part, int npq,
                                                    double* __restrict__ part, int par) {
  __shared__ double s_red[kBS / 64];
  if (ks->done) return;
  const double pq = dev::sum_partials<kBS>(pq_part, npq, 1, s_red);
  const double a = ks->rho2[par ^ 1] / pq;
  const float alpha = (float)a;
  if (blockIdx.x == 0 && threadIdx.x == 0) ks->alpha2[par ^ 1] = a;
  double rr = 0.0;
  for (int64_t q = (int64_t)blockIdx.x * kBS + threadIdx.x; q < n; q += (int64_t)gridDim.x * kBS) {
    const float ri = fmaf(-alpha, __builtin_nontemporal_load(&ap[q]), r[q]);
    r[q] = ri;
    rr += (double)ri * (double)ri;
  }
  rr = dev::block_sum<kBS>(rr, s_red);
  if (threadIdx.x == 0) part[blockIdx.x] = rr;
}

dim3 grid_of(const MgGrid& g) {
  return dim3((unsigned)((g.pitch + 63) / 64), (unsigned)((g.cy + 4) / 4), (unsigned)(g.cz + 1));
}

// Builds the hierarchy for the context's current operator; false where it does not apply:
// a system loaded as CSR, a mesh that is not an octree of cubes on one lattice of at most
// 1022 cells an axis, Dirichlet nodes other than the box faces, or a mesh so sparse on
// its finest lattice that the dense transfer array would cost more than the iterations it
// saves.
bool build_hierarchy(ngpb_ctx* c) {
  if (c->external_csr || !c->have_mesh || c->n != c->N || c->L <= 0 || c->n < 64) return false;
  const MeshView m = mesh_view_of(c);
  const int64_t n = c->n, L = c->L;
  hipStream_t st = c->stream;
  DBuf<int> bad(st);
  bad.resize(1);
  NGPB_HIP(hipMemsetAsync(bad.p, 0, sizeof(int), st));
  int hb = 0;
  auto is_bad = [&] {
    NGPB_HIP(hipGetLastError());
    NGPB_HIP(hipMemcpyAsync(&hb, bad.p, sizeof(int), hipMemcpyDeviceToHost, st));
    NGPB_HIP(hipStreamSynchronize(st));
    return hb != 0;
  };
  MgBox g;
  {
    const unsigned gb = (unsigned)std::min<int64_t>(1024, blocks_for(std::max(L, n), kBS));
    DBuf<double> part(st);
    part.resize((size_t)7 * gb);
    hipLaunchKernelGGL(k_mg_extent, dim3(gb), dim3(kBS), 0, st, m, part.p, bad.p);
    std::vector<double> h((size_t)7 * gb);
    NGPB_HIP(hipMemcpyAsync(h.data(), part.p, h.size() * sizeof(double), hipMemcpyDeviceToHost, st));
    if (is_bad()) return false;
    double e = INFINITY, lo[3] = {INFINITY, INFINITY, INFINITY}, hi[3] = {-INFINITY, -INFINITY, -INFINITY};
    for (unsigned k = 0; k < gb; ++k) {
      e = std::min(e, h[7 * k]);
      for (int d = 0; d < 3; ++d) {
        lo[d] = std::min(lo[d], h[7 * k + 1 + d]);
        hi[d] = std::max(hi[d], h[7 * k + 4 + d]);
      }
    }
    if (!(e > 0.0) || !std::isfinite(e)) return false;
    for (int d = 0; d < 3; ++d) {
      const double u = (hi[d] - lo[d]) / e;
      if (!(u >= 3.0 - 1e-3) || !(u <= 1022.0) || std::fabs(u - std::rint(u)) > 1e-3) return false;
      g.x0[d] = lo[d];
      g.n[d] = (int)std::rint(u);
    }
    // the spacing from the longest axis: the mesh's own rounding of its coordinates
    const int d = (int)(std::max_element(g.n, g.n + 3) - g.n);
    g.h = (hi[d] - lo[d]) / g.n[d];
    g.inv_h = 1.0 / g.h;
  }
  MgHierarchy& H = c->mg;
  H = MgHierarchy();
  H.dpitch = (g.n[0] + 1 + 3) / 4 * 4;
  H.drows = g.n[1] + 1;
  const int64_t dense = (int64_t)H.dpitch * H.drows * (g.n[2] + 1);
  if (dense > kMgDenseRatio * n || dense >= ((int64_t)1 << 31)) return false;
  int cells[3] = {g.n[0], g.n[1], g.n[2]};
  int64_t floats = 0;
  while (H.nlev < kMgLevels) {
    for (int d = 0; d < 3; ++d) cells[d] = (cells[d] + 1) / 2;
    MgGrid& l = H.lev[H.nlev++];
    l.cx = cells[0];
    l.cy = cells[1];
    l.cz = cells[2];
    l.pitch = (l.cx + 1 + 3) / 4 * 4;
    floats += l.nodes() * 8;  // ex ey ez dinv b x t f
    if (std::min({cells[0], cells[1], cells[2]}) <= 2) break;
  }
  auto take = [&](auto& buf, int64_t count) {
    buf.reserve((size_t)count);
    if (c->mg_max_bytes > 0 && c->mg_bytes() > c->mg_max_bytes)
      throw Error(NGPB_E_NOMEM, "the multigrid hierarchy exceeds its memory bound");
  };
  take(c->mg_pool, floats);
  take(c->mg_dense, dense);
  take(c->mg_pos, n);
  take(c->mg_sd, n);
  take(c->mg_r, n + 2 * kGuard);
  take(c->mg_z, n + 2 * kGuard);
  H.dense = c->mg_dense.p;
  {
    float* p = c->mg_pool.p;
    for (int l = 0; l < H.nlev; ++l) {
      MgGrid& q = H.lev[l];
      const int64_t cnt = q.nodes();
      for (float** a : {&q.ex, &q.ey, &q.ez, &q.dinv, &q.b, &q.x, &q.t, &q.f}) {
        *a = p;
        p += cnt;
      }
      if (l < 1 || l > 3) q.f = nullptr;  // direct nodes live on levels 2, 3 and 4
    }
  }
  const int max_direct = std::min(3, H.nlev - 1);
  DBuf<uint8_t> level(st), nlev(st);
  level.resize((size_t)L);
  nlev.resize((size_t)n);
  // the dense array holds the leaf map during the setup (one 4-byte entry per cell)
  int32_t* map = reinterpret_cast<int32_t*>(c->mg_dense.p);
  NGPB_HIP(hipMemsetAsync(map, 0xff, (size_t)dense * 4, st));
  NGPB_HIP(hipMemsetAsync(nlev.p, 0xff, (size_t)n, st));
  hipLaunchKernelGGL(k_mg_leaf_map, dim3(blocks_for(L, kBS)), dim3(kBS), 0, st, m, g, map, level.p, bad.p);
  if (is_bad()) return false;  // levels of a mesh off the lattice are not set
  for (int s = max_direct + 1; s >= 2; --s)
    hipLaunchKernelGGL(k_mg_node_level, dim3(blocks_for(L, kBS)), dim3(kBS), 0, st, L, c->leaf_corner.p, level.p, s,
                       s == max_direct + 1 ? 31 : s, nlev.p);
  hipLaunchKernelGGL(k_mg_node_level, dim3(blocks_for(L, kBS)), dim3(kBS), 0, st, L, c->leaf_corner.p, level.p, 0,
                     max_direct == 0 ? 31 : 1, nlev.p);
  hipLaunchKernelGGL(k_mg_rows, dim3(blocks_for(n, kBS)), dim3(kBS), 0, st, n, c->node_xyz.p, g, c->rowptr.p,
                     c->dscale.p, c->sell_banded ? c->row_perm.p : nullptr, nlev.p, max_direct, c->mg_pos.p,
                     c->mg_sd.p, bad.p);
  DBuf<float4> ca(st), cb(st);
  {
    const MgGrid& l = H.lev[0];
    const int64_t nc = (int64_t)l.cx * l.cy * l.cz;
    ca.resize((size_t)nc);
    cb.resize((size_t)(nc / 8 + 2 * (int64_t)(l.cx + 2) * (l.cy + 2) + 2 * (int64_t)(l.cz + 2) * (l.cx + l.cy + 4)));
    hipLaunchKernelGGL(k_mg_cells1, dim3(blocks_for(8 * nc, kBS)), dim3(kBS), 0, st, m, g, l.cx, l.cy, l.cz, map, level.p,
                       c->c_edge.p, c->reac.p, ca.p, bad.p);
  }
  if (is_bad()) return false;
  NGPB_HIP(hipMemsetAsync(c->mg_dense.p, 0, (size_t)dense * 4, st));
  for (int l = 0; l < H.nlev; ++l) {
    const MgGrid& q = H.lev[l];
    if (l > 0) {
      const MgGrid& f = H.lev[l - 1];
      const int64_t nc = (int64_t)q.cx * q.cy * q.cz;
      NGPB_REQUIRE((size_t)nc <= cb.n, NGPB_E_STATE, "multigrid cell buffer too small");
      hipLaunchKernelGGL(k_mg_cells, dim3(blocks_for(nc, kBS)), dim3(kBS), 0, st, f.cx, f.cy, f.cz, ca.p, q.cx, q.cy,
                         q.cz, cb.p);
      ca.swap(cb);
    }
    hipLaunchKernelGGL(k_mg_edges, grid_of(q), dim3(kBS), 0, st, q, (float)(g.h * (double)(2 << l)), ca.p);
    // after the first swap both buffers hold at least an eighth of level 1's cells
  }
  NGPB_HIP(hipGetLastError());
  // the bottom kernel takes the levels that fit one block
  H.bottom = mg_bottom_level(H);
  if (H.bottom < 0) return false;
  NGPB_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(k_mg_bottom), hipFuncAttributeMaxDynamicSharedMemorySize,
                               kMgBottomLds));
  NGPB_HIP(hipStreamSynchronize(st));
  return true;
}

}  // namespace

void mg_release(ngpb_ctx* c) {
  c->mg_pool.release();
  c->mg_dense.release();
  c->mg_sd.release();
  c->mg_r.release();
  c->mg_z.release();
  c->mg_pos.release();
  c->mg = MgHierarchy();
}

// True once the hierarchy of the current operator is built, false (c->mg_state = -1) where
// it does not apply or there is no memory for it: the solve then uses Jacobi scaling, and
// nothing is held.
bool mg_setup(ngpb_ctx* c) {
  if (c->mg_state) return c->mg_state > 0;
  c->mg_state = -1;
  bool ok = false;
  try {
    ok = c->mg_cycle_iters > 0 && build_hierarchy(c);
  } catch (const Error& e) {
    mg_release(c);
    if (e.code != NGPB_E_NOMEM) throw;
  } catch (...) {
    mg_release(c);
    throw;
  }
  if (ok) c->mg_state = 1;
  else mg_release(c);
  return ok;
}

// ------------------------------------------------------------------ launches
void mg_precondition(ngpb_ctx* c, const float* r, const float* ar, float* z, const double* rr_part, int npr,
                     double* rz_part, int par, bool first) {
  const MgHierarchy& H = c->mg;
  const int64_t n = c->n;
  const unsigned gv = vec_grid(n);
  hipStream_t st = c->stream;
  KrylovScalars* ks = c->ks.p;
  hipLaunchKernelGGL(k_mgf_embed, dim3(gv), dim3(kBS), 0, st, H, n, c->mg_pos.p, c->mg_sd.p, r, ar, ks, rr_part, npr,
                     par, first ? 1 : 0);
  for (int l = 0; l <= H.bottom; ++l) {
    const MgGrid& q = H.lev[l];
    const dim3 gp(blocks_for(mg_pairs(q), kBS));
    if (l == 0)
      hipLaunchKernelGGL(k_mg_restrict, gp, dim3(kBS), 0, st, q, H.dense, H.dpitch, H.drows, ks);
    else
      hipLaunchKernelGGL(k_mg_restrict, gp, dim3(kBS), 0, st, q, H.lev[l - 1].t, H.lev[l - 1].pitch,
                         H.lev[l - 1].cy + 1, ks);
    if (l < H.bottom) hipLaunchKernelGGL(k_mg_resid, dim3(blocks_for(mg_quads(q), kBS)), dim3(kBS), 0, st, q, ks);
  }
  hipLaunchKernelGGL(k_mg_bottom, dim3(1), dim3(kMgBottomBS), (unsigned)mg_bottom_lds(H, H.bottom), st, H, ks);
  for (int l = H.bottom - 1; l >= 0; --l) {
    const dim3 gq(blocks_for(mg_quads(H.lev[l]), kBS));
    hipLaunchKernelGGL(k_mg_prolong, gq, dim3(kBS), 0, st, H.lev[l], H.lev[l + 1], ks);
    hipLaunchKernelGGL(k_mg_smooth, gq, dim3(kBS), 0, st, H.lev[l], ks);
  }
  hipLaunchKernelGGL(k_mgf_correct, dim3(gv), dim3(kBS), 0, st, H, n, c->mg_pos.p, c->mg_sd.p, r, ar, z, ks, rz_part);
}

void mg_direction(ngpb_ctx* c, const float* r, const float* az, const float* z, float* p, float* x,
                  const double* rz_part, int par) {
  const int64_t n = c->n;
  const unsigned gv = vec_grid(n);
  hipLaunchKernelGGL(k_mgf_dir, dim3(gv), dim3(kBS), 0, c->stream, n, z, r, az, p, x, c->ks.p, rz_part, (int)gv, par);
}

void mg_update(ngpb_ctx* c, float* r, const float* ap, const double* pq_part, int npq, double* part, int par) {
  const int64_t n = c->n;
  hipLaunchKernelGGL(k_mgf_update, dim3(vec_grid(n)), dim3(kBS), 0, c->stream, n, r, ap, c->ks.p, pq_part, npq, part,
                     par);
}

}  // namespace ngpb
