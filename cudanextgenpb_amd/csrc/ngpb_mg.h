// Data of the multigrid preconditioner (ngpb_mg.hip).
#pragma once
#include <hip/hip_runtime.h>

#include <cstdint>

namespace ngpb {

constexpr int kMgLevels = 10;  // 1022 cells an axis halve nine times
// Finest-lattice vertices per unknown up to which the dense transfer array is used. An
// iteration then moves some 4 x 32 bytes for it and 2 x 32 for the uniform levels per
// unknown, ~450 with the three SpMVs, against ~60 for a Jacobi-scaled one of which there
// are ten or more times as many: at 18 per unknown (a 47,302-unknown mesh) the solve is
// still 1.5x faster, at 24 (706,224 unknowns) 5.9 ms for 12.5. The bound is on memory: at 32
// the hierarchy takes some 290 bytes per unknown.
constexpr int64_t kMgDenseRatio = 32;
// the finest lattice of the mesh's box
struct MgBox {
  double x0[3] = {0, 0, 0};
  double h = 0, inv_h = 0;
  int n[3] = {0, 0, 0};  // cells
};

// A uniform level of cx x cy x cz cells: nodes 0 .. c per axis, x fastest, rows of `pitch`.
struct MgGrid {
  int cx = 0, cy = 0, cz = 0, pitch = 0;
  float *ex = nullptr, *ey = nullptr, *ez = nullptr;  // conductance to the next node along the axis
  float* dinv = nullptr;                              // inverse diagonal, 0 on the faces
  float *b = nullptr, *x = nullptr, *t = nullptr;     // right-hand side, iterate, residual / result
  float* f = nullptr;                                 // residual of the octree nodes that live on this level
  __host__ __device__ int64_t nodes() const { return (int64_t)pitch * (cy + 1) * (cz + 1); }
  __device__ __forceinline__ int64_t at(int i, int j, int k) const {
    return ((int64_t)k * (cy + 1) + j) * pitch + i;
  }
  __device__ __forceinline__ bool inner(int i, int j, int k) const {
    return i > 0 && i < cx && j > 0 && j < cy && k > 0 && k < cz;
  }
};

struct MgHierarchy {
  int nlev = 0;    // uniform levels; lev[l] has spacing 2^(l + 1) hf
  int bottom = 0;  // first level of the one-block bottom kernel
  int dpitch = 0, drows = 0;
  float* dense = nullptr;  // residual on the finest lattice
  MgGrid lev[kMgLevels];
};

}  // namespace ngpb
