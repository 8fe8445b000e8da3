// Device bodies of the multigrid cycle, shared by the single-system and the batched
// solvers: both evaluate a level with the same instructions in the same order.
#pragma once
#include <type_traits>

#include "ngpb_internal.h"

namespace ngpb {
namespace {

// damping of the Jacobi smoother (22 and 27 iterations at 0.9, 23 and 28 at 0.8 on a
// ligand and a 300-atom globule)
constexpr float kMgOmega = 0.9f;
constexpr int kMgBottomBS = 1024;
constexpr int kMgBottomPer = 4;     // nodes per thread on the bottom kernel's first level
constexpr int kMgBottomDepth = 6;   // levels it takes at most
constexpr int kMgBottomLds = 96 * 1024;

// threads of the level kernels
__host__ __device__ inline int mg_quads(const MgGrid& g) { return g.pitch / 4 * (g.cy - 1) * (g.cz - 1); }
__host__ __device__ inline int mg_pairs(const MgGrid& g) { return g.pitch / 2 * (g.cy - 1) * (g.cz - 1); }
inline int mg_bottom_lds(const MgHierarchy& h, int first) {
  int64_t n = 0;
  for (int l = first; l < h.nlev; ++l) n += h.lev[l].nodes();
  return (int)std::min<int64_t>(n * 2 * (int64_t)sizeof(float), INT32_MAX);
}

// First level of the bottom kernel, -1 if none fits: its levels after the first have at
// most one interior node per thread, the first kMgBottomPer.
inline int mg_bottom_level(const MgHierarchy& h) {
  auto inner = [&](int l) {
    return (int64_t)(h.lev[l].cx - 1) * (h.lev[l].cy - 1) * (h.lev[l].cz - 1);
  };
  int first = -1;
  for (int l = h.nlev - 1; l >= 0 && h.nlev - l <= kMgBottomDepth; --l) {
    if (inner(l) > (int64_t)kMgBottomPer * kMgBottomBS || mg_bottom_lds(h, l) > kMgBottomLds) break;
    first = l;
    if (inner(l) > kMgBottomBS) break;
  }
  return first;
}

// row of a quad or pair index: the interior rows of the grid, one after another
__device__ __forceinline__ bool mg_row(const MgGrid& g, int t, int per, int* q, int* j, int* k) {
  const int r = t / per;
  *q = t - r * per;
  *k = r / (g.cy - 1) + 1;
  *j = r - (*k - 1) * (g.cy - 1) + 1;
  return *k < g.cz;
}

// sum of conductance times neighbour over the six neighbours, of four nodes from o on
__device__ __forceinline__ float4 mg_nb_quad(const MgGrid& g, const float* __restrict__ v, int64_t o) {
  const int64_t sy = g.pitch, sz = (int64_t)g.pitch * (g.cy + 1);
  auto ld = [](const float* p) { return *reinterpret_cast<const float4*>(p); };
  const float4 c = ld(v + o), ex = ld(g.ex + o);
  const float vl = v[o - 1], vr = v[o + 4], el = g.ex[o - 1];
  const float4 ey = ld(g.ey + o), eym = ld(g.ey + o - sy), ez = ld(g.ez + o), ezm = ld(g.ez + o - sz);
  const float4 yp = ld(v + o + sy), ym = ld(v + o - sy), zp = ld(v + o + sz), zm = ld(v + o - sz);
  float4 s;
  s.x = ex.x * c.y + el * vl;
  s.y = ex.y * c.z + ex.x * c.x;
  s.z = ex.z * c.w + ex.y * c.y;
  s.w = ex.w * vr + ex.z * c.z;
  auto add = [](float4& a, const float4& p, const float4& q) {
    a.x = fmaf(p.x, q.x, a.x);
    a.y = fmaf(p.y, q.y, a.y);
    a.z = fmaf(p.z, q.z, a.z);
    a.w = fmaf(p.w, q.w, a.w);
  };
  add(s, ey, yp);
  add(s, eym, ym);
  add(s, ez, zp);
  add(s, ezm, zm);
  return s;
}

// keeps the interior nodes of a quad at i, zero elsewhere
__device__ __forceinline__ float4 mg_mask(const MgGrid& g, int i, float4 v) {
  if (i == 0) v.x = 0.f;
  if (i >= g.cx) v.x = 0.f;
  if (i + 1 >= g.cx) v.y = 0.f;
  if (i + 2 >= g.cx) v.z = 0.f;
  if (i + 3 >= g.cx) v.w = 0.f;
  return v;
}

// residual after the first smoothing step x = omega b / d: t = b - A x. Four nodes a
// thread with 16-byte accesses: 14 loads instead of 52 (level 1 of the 8M-node mesh, 2.2M
// nodes: 22 us with a node a thread).
__device__ __forceinline__ void mg_resid_quad(const MgGrid& g, int t) {
  int q, j, k;
  if (!mg_row(g, t, g.pitch / 4, &q, &j, &k)) return;
  const int64_t o = g.at(4 * q, j, k);
  const float4 s = mg_nb_quad(g, g.x, o), b = *reinterpret_cast<const float4*>(g.b + o);
  float4 r;
  r.x = fmaf(1.f - kMgOmega, b.x, s.x);
  r.y = fmaf(1.f - kMgOmega, b.y, s.y);
  r.z = fmaf(1.f - kMgOmega, b.z, s.z);
  r.w = fmaf(1.f - kMgOmega, b.w, s.w);
  *reinterpret_cast<float4*>(g.t + o) = mg_mask(g, 4 * q, r);
}

// second smoothing step: t = x + omega (b - A x) / d
__device__ __forceinline__ void mg_smooth_quad(const MgGrid& g, int t) {
  int q, j, k;
  if (!mg_row(g, t, g.pitch / 4, &q, &j, &k)) return;
  const int64_t o = g.at(4 * q, j, k);
  auto ld = [](const float* p) { return *reinterpret_cast<const float4*>(p); };
  const float4 s = mg_nb_quad(g, g.x, o), b = ld(g.b + o), x = ld(g.x + o), d = ld(g.dinv + o);
  float4 r;  // d = 0 and x = 0 off the interior
  r.x = fmaf(1.f - kMgOmega, x.x, kMgOmega * d.x * (b.x + s.x));
  r.y = fmaf(1.f - kMgOmega, x.y, kMgOmega * d.y * (b.y + s.y));
  r.z = fmaf(1.f - kMgOmega, x.z, kMgOmega * d.z * (b.z + s.z));
  r.w = fmaf(1.f - kMgOmega, x.w, kMgOmega * d.w * (b.w + s.w));
  *reinterpret_cast<float4*>(g.t + o) = r;
}

// b = R t + f, x = omega b / d: full weighting of t (rows of `pitch`, `rows` rows per
// plane) around fine nodes (2i, 2j, 2k), two coarse nodes a thread from 16-byte loads.
// Every index read is inside the fine array for an interior row.
__device__ __forceinline__ void mg_restrict_pair(const MgGrid& g, const float* __restrict__ t, int pitch, int rows,
                                                 int at) {
  int q, j, k;
  if (!mg_row(g, at, g.pitch / 2, &q, &j, &k)) return;
  const int i = 2 * q;
  if (i >= g.cx) return;
  const int64_t o = g.at(i, j, k);
  float s0 = 0.f, s1 = 0.f;
#pragma unroll
  for (int dk = -1; dk <= 1; ++dk) {
#pragma unroll
    for (int dj = -1; dj <= 1; ++dj) {
      const float* r = t + ((int64_t)(2 * k + dk) * rows + 2 * j + dj) * pitch + 4 * q;
      // row ends: entries past the row belong to the next row and count for face nodes only
      const float4 v = *reinterpret_cast<const float4*>(r);
      const float w = (dk ? 0.5f : 1.f) * (dj ? 0.5f : 1.f);
      s0 = fmaf(w, fmaf(0.5f, r[-1] + v.y, v.x), s0);
      s1 = fmaf(w, fmaf(0.5f, v.y + v.w, v.z), s1);
    }
  }
  if (g.f) {
    s0 += g.f[o];
    s1 += g.f[o + 1];
  }
  if (i == 0) s0 = 0.f;
  if (i + 1 >= g.cx) s1 = 0.f;
  *reinterpret_cast<float2*>(g.b + o) = make_float2(s0, s1);
  const float2 d = *reinterpret_cast<const float2*>(g.dinv + o);
  *reinterpret_cast<float2*>(g.x + o) = make_float2(kMgOmega * d.x * s0, kMgOmega * d.y * s1);
}

// x += trilinear interpolation of the coarse level's result
__device__ __forceinline__ void mg_prolong_quad(const MgGrid& g, const MgGrid& c, int t) {
  int q, j, k;
  if (!mg_row(g, t, g.pitch / 4, &q, &j, &k)) return;
  const int i = 4 * q;
  if (i >= g.cx) return;
  const int64_t o = g.at(i, j, k);
  float a = 0.f, b = 0.f, d = 0.f;  // coarse values at 2q, 2q + 1, 2q + 2 on this row
  const int J = j >> 1, K = k >> 1, jo = j & 1, ko = k & 1;
  const float w = (jo ? 0.5f : 1.f) * (ko ? 0.5f : 1.f);
  const int last = c.pitch - 1;
  for (int z = 0; z <= ko; ++z)
    for (int y = 0; y <= jo; ++y) {
      const float* r = c.t + c.at(0, J + y, K + z);
      a = fmaf(w, r[min(2 * q, last)], a);
      b = fmaf(w, r[min(2 * q + 1, last)], b);
      d = fmaf(w, r[min(2 * q + 2, last)], d);
    }
  float4 x = *reinterpret_cast<const float4*>(g.x + o);
  x.x += a;
  x.y += 0.5f * (a + b);
  x.z += b;
  x.w += 0.5f * (b + d);
  *reinterpret_cast<float4*>(g.x + o) = mg_mask(g, i, x);
}

// trilinear interpolation of values e at fine position (i, j, k)
template <class At>
__device__ __forceinline__ float mg_interpolate(int i, int j, int k, At&& e) {
  const int I = i >> 1, J = j >> 1, K = k >> 1, a = i & 1, b = j & 1, c = k & 1;
  auto ex = [&](int y, int z) { return a ? 0.5f * (e(I, y, z) + e(I + 1, y, z)) : e(I, y, z); };
  auto ey = [&](int z) { return b ? 0.5f * (ex(J, z) + ex(J + 1, z)) : ex(J, z); };
  return c ? 0.5f * (ey(K) + ey(K + 1)) : ey(K);
}

// The levels from h.bottom on, one cycle in one block of kMgBottomBS threads. A thread
// keeps its nodes' coefficients and right-hand sides in registers, loaded at the start
// all at once; x and t of every level are in LDS. (Loading the coefficients stage by
// stage from memory, the kernel took 29 us from an 18^3-node level on: ~20 stages, each
// with the latency of a memory read.) The last level has one interior node (solved
// exactly) or, in a flat box, a few lines of them (16 steps).
struct MgBottomNode {
  float xm, xp, ym, yp, zm, zp, d, b;
  int o, i, j, k;
};

__device__ __forceinline__ void mg_bottom(const MgHierarchy& h, float* s_mem) {
  const int first = h.bottom, depth = h.nlev - first;
  const int tid = threadIdx.x;
  float *xs[kMgBottomDepth], *ts[kMgBottomDepth];
  {
    float* p = s_mem;
#pragma unroll
    for (int s = 0; s < kMgBottomDepth; ++s) {
      xs[s] = ts[s] = s_mem;
      if (s < depth) {
        const int cnt = (int)h.lev[first + s].nodes();
        xs[s] = p;
        ts[s] = p + cnt;
        p += 2 * cnt;
      }
    }
    for (int q = tid; q < (int)(p - s_mem); q += kMgBottomBS) s_mem[q] = 0.f;
  }
  // interior node q of a level; o < 0: none
  auto node = [&](const MgGrid& g, int q) {
    MgBottomNode m{};
    m.o = -1;
    const int nx = g.cx - 1, ny = g.cy - 1;
    if (q >= nx * ny * (g.cz - 1)) return m;
    const int r = q / nx;
    m.i = q - r * nx + 1;
    m.k = r / ny + 1;
    m.j = r - (m.k - 1) * ny + 1;
    const int64_t o = g.at(m.i, m.j, m.k);
    m.o = (int)o;
    m.xp = g.ex[o];
    m.xm = g.ex[o - 1];
    m.yp = g.ey[o];
    m.ym = g.ey[o - g.pitch];
    m.zp = g.ez[o];
    m.zm = g.ez[o - g.pitch * (g.cy + 1)];
    m.d = g.dinv[o];
    return m;
  };
  MgBottomNode n0[kMgBottomPer], nl[kMgBottomDepth];
#pragma unroll
  for (int u = 0; u < kMgBottomPer; ++u) {
    n0[u] = node(h.lev[first], u * kMgBottomBS + tid);
    if (n0[u].o >= 0) n0[u].b = h.lev[first].b[n0[u].o];
  }
#pragma unroll
  for (int s = 1; s < kMgBottomDepth; ++s) {
    nl[s].o = -1;
    if (s >= depth) continue;
    const MgGrid& g = h.lev[first + s];
    nl[s] = node(g, tid);
    if (nl[s].o >= 0 && g.f) nl[s].b = g.f[nl[s].o];
  }
  auto nb = [&](const MgGrid& g, const MgBottomNode& m, const float* v) {
    const int sy = g.pitch, sz = g.pitch * (g.cy + 1), o = m.o;
    return m.xp * v[o + 1] + m.xm * v[o - 1] + m.yp * v[o + sy] + m.ym * v[o - sy] + m.zp * v[o + sz] +
           m.zm * v[o - sz];
  };
  // the nodes of level s that this thread owns
  auto each = [&](auto s_, auto&& fn) {
    constexpr int s = decltype(s_)::value;
    if constexpr (s == 0) {
#pragma unroll
      for (int u = 0; u < kMgBottomPer; ++u)
        if (n0[u].o >= 0) fn(n0[u]);
    } else {
      if (nl[s].o >= 0) fn(nl[s]);
    }
  };
  __syncthreads();
  each(std::integral_constant<int, 0>(), [&](MgBottomNode& m) { xs[0][m.o] = kMgOmega * m.d * m.b; });
  __syncthreads();
  auto down = [&](auto s_) {  // level s to level s + 1
    constexpr int s = decltype(s_)::value;
    if (s + 1 >= depth) return;
    const MgGrid &g = h.lev[first + s], &c = h.lev[first + s + 1];
    const float* x = xs[s];
    float* t = ts[s];
    each(s_, [&](MgBottomNode& m) { t[m.o] = fmaf(1.f - kMgOmega, m.b, nb(g, m, x)); });
    __syncthreads();
    const int rows = g.cy + 1, pitch = g.pitch;
    float* xc = xs[s + 1];
    each(std::integral_constant<int, s + 1>(), [&](MgBottomNode& m) {
      float b = 0.f;
#pragma unroll
      for (int dk = -1; dk <= 1; ++dk)
#pragma unroll
        for (int dj = -1; dj <= 1; ++dj) {
          const float* r = t + ((2 * m.k + dk) * rows + 2 * m.j + dj) * pitch + 2 * m.i;
          const float w = (dk ? 0.5f : 1.f) * (dj ? 0.5f : 1.f);
          b = fmaf(w, fmaf(0.5f, r[-1] + r[1], r[0]), b);
        }
      m.b += b;  // f before
      xc[m.o] = kMgOmega * m.d * m.b;
    });
    __syncthreads();
  };
  auto last = [&](auto s_) {
    constexpr int s = decltype(s_)::value;
    if (s + 1 != depth) return;
    const MgGrid& g = h.lev[first + s];
    float *x = xs[s], *t = ts[s];
    if ((g.cx - 1) * (g.cy - 1) * (g.cz - 1) == 1) {
      each(s_, [&](MgBottomNode& m) { t[m.o] = m.d * m.b; });
      __syncthreads();
      return;
    }
    for (int it = 0; it < 15; ++it) {  // x holds the first step; the 16th ends in t
      const float* from = it & 1 ? t : x;
      float* to = it & 1 ? x : t;
      each(s_, [&](MgBottomNode& m) {
        to[m.o] = fmaf(1.f - kMgOmega, from[m.o], kMgOmega * m.d * (m.b + nb(g, m, from)));
      });
      __syncthreads();
    }
  };
  auto up = [&](auto s_) {  // level s + 1 to level s
    constexpr int s = decltype(s_)::value;
    if (s + 1 >= depth) return;
    const MgGrid &g = h.lev[first + s], &c = h.lev[first + s + 1];
    float *x = xs[s], *t = ts[s];
    const float* e = ts[s + 1];
    each(s_, [&](MgBottomNode& m) {
      x[m.o] += mg_interpolate(m.i, m.j, m.k, [&](int a, int b, int d) { return e[c.at(a, b, d)]; });
    });
    __syncthreads();
    each(s_, [&](MgBottomNode& m) {
      t[m.o] = fmaf(1.f - kMgOmega, x[m.o], kMgOmega * m.d * (m.b + nb(g, m, x)));
    });
    __syncthreads();
  };
  using std::integral_constant;
  down(integral_constant<int, 0>());
  down(integral_constant<int, 1>());
  down(integral_constant<int, 2>());
  down(integral_constant<int, 3>());
  down(integral_constant<int, 4>());
  last(integral_constant<int, 0>());
  last(integral_constant<int, 1>());
  last(integral_constant<int, 2>());
  last(integral_constant<int, 3>());
  last(integral_constant<int, 4>());
  last(integral_constant<int, 5>());
  up(integral_constant<int, 4>());
  up(integral_constant<int, 3>());
  up(integral_constant<int, 2>());
  up(integral_constant<int, 1>());
  up(integral_constant<int, 0>());
  // results that kernels outside read: the first level, and levels with direct nodes
  each(integral_constant<int, 0>(), [&](MgBottomNode& m) { h.lev[first].t[m.o] = ts[0][m.o]; });
  auto out = [&](auto s_) {
    constexpr int s = decltype(s_)::value;
    if (s >= depth || !h.lev[first + s].f) return;
    each(s_, [&](MgBottomNode& m) { h.lev[first + s].t[m.o] = ts[s][m.o]; });
  };
  out(integral_constant<int, 1>());
  out(integral_constant<int, 2>());
  out(integral_constant<int, 3>());
}

// ---- octree rows: pos packs a row's position (10 bits per axis) and its level
__device__ __forceinline__ void mg_embed(const MgHierarchy& h, uint32_t p, float v) {
  const int i = p & 1023, j = (p >> 10) & 1023, k = (p >> 20) & 1023, d = p >> 30;
  if (d == 0) {
    h.dense[((int64_t)k * h.drows + j) * h.dpitch + i] = v;
  } else {
    const MgGrid& g = h.lev[d];  // level d + 1
    g.f[g.at(i >> (d + 1), j >> (d + 1), k >> (d + 1))] = v;
  }
}

// Coarse correction at a row's position; called by whole waves. Rows of a run along x
// share coarse values: a lane loads the one at or above it, and a lane at an odd
// position takes the one below from its left neighbour, if that is the row before.
__device__ __forceinline__ float mg_correction(const MgHierarchy& h, uint32_t p, bool valid) {
  const int i = p & 1023, j = (p >> 10) & 1023, k = (p >> 20) & 1023, d = p >> 30;
  const uint32_t left = (uint32_t)__builtin_amdgcn_update_dpp((int)0xffffffff, (int)p, 0x138, 0xf, 0xf, false);
  const bool run = (i & 1) && left + 1 == p;
  float e = 0.f;
  if (d == 0) {
    const MgGrid& g = h.lev[0];
    const int J = j >> 1, K = k >> 1, jo = j & 1, ko = k & 1;
    const float w = (jo ? 0.5f : 1.f) * (ko ? 0.5f : 1.f);
    float hi = 0.f, lo = 0.f;
    if (valid) {
      const int I = min((i + 1) >> 1, g.cx);
      for (int z = 0; z <= ko; ++z)
        for (int y = 0; y <= jo; ++y) {
          const float* r = g.t + g.at(0, min(J + y, g.cy), min(K + z, g.cz));
          hi = fmaf(w, r[I], hi);
          if ((i & 1) && !run) lo = fmaf(w, r[i >> 1], lo);
        }
    }
    const float below = __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(hi), 0x138, 0xf, 0xf, false));
    e = (i & 1) ? 0.5f * (hi + (run ? below : lo)) : hi;
  } else if (valid) {
    const MgGrid& g = h.lev[d];
    e = g.t[g.at(i >> (d + 1), j >> (d + 1), k >> (d + 1))];
  }
  return e;
}

}  // namespace
}  // namespace ngpb
