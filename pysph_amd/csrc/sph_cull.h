// Stencil rows culled to a destination's search sphere, shared by the packed
// FP32 scans and the group scan of the SoA passes.
#pragma once
#include "sph_common.h"

namespace sph {

// ---------------------------------------------------------------------------
// stencil rows with geometric culling
// ---------------------------------------------------------------------------
struct Cull {
  float xd, yd, zd, rc2, r;
};

// Distance from v to the extent of cell c along one axis; border cells
// reach to infinity because the binning clamps outside particles into them.
__device__ __forceinline__ float axis_gap(float v, int c, int n, int lo, float cs) {
  float gap = 0.f;
  if (c > 0) gap = fmaxf(gap, (float)(c + lo) * cs - v);
  if (c < n - 1) gap = fmaxf(gap, v - (float)(c + lo + 1) * cs);
  return gap;
}

// rc is widened for FP32 rounding of positions and cell boundaries.
__device__ __forceinline__ Cull make_cull(const float4& pd, double rc, const Grid& g) {
  Cull c;
  c.xd = pd.x;
  c.yd = pd.y;
  c.zd = pd.z;
  const float scale = fabsf(pd.x) + fabsf(pd.y) + fabsf(pd.z) + g.cs_f;
  const float r = (float)rc * 1.00001f + 8e-7f * scale;
  c.rc2 = r * r;
  c.r = r;
  return c;
}

// The cull runs in FP32 (its radius carries the margin for that); points,
// radii or cells outside its range take the whole ring.
__device__ __forceinline__ bool can_cull(const Grid& g, double x, double y, double z, double rc) {
  return fabs(x) + fabs(y) + fabs(z) < 1e30 && fabs(rc) < 1e15 && g.cs > 1e-15 && g.cs < 1e15;
}

// Stencil offsets [a, b] (within +-ring) along one axis whose cells can
// hold a point within the cull radius of v; border cells reach to infinity.
// The margin of the cull radius covers the FP32 rounding of the bounds, as
// in row_range_cull.
__device__ __forceinline__ void axis_span(float v, float r, int c, int n, int lo, float inv_cs,
                                          int ring, int& a, int& b) {
  const float last = (float)(n - 1);
  const float fa = fminf(fmaxf(floorf((v - r) * inv_cs) - (float)lo, 0.f), last);
  const float fb = fminf(fmaxf(floorf((v + r) * inv_cs) - (float)lo, 0.f), last);
  if (!(fa <= fb)) {  // NaN positions keep the ring
    a = -ring;
    b = ring;
    return;
  }
  a = max((int)fa - c, -ring);
  b = min((int)fb - c, ring);
}

// Cells of grid row (y, z) within the stencil ring of cell column cx whose
// extent can hold a point within the cull radius, as cell-start indices
// [k0, k1] (read cstart[k0] and cstart[k1]); false when there is none.
__device__ __forceinline__ bool row_cells_cull(const Grid& g, int cx, int y, int z, int ring,
                                               const Cull& cu, int& k0, int& k1) {
  if (y < 0 || y >= g.dims[1] || z < 0 || z >= g.dims[2]) return false;
  const float gy = axis_gap(cu.yd, y, g.dims[1], g.lo[1], g.cs_f);
  const float gz = axis_gap(cu.zd, z, g.dims[2], g.lo[2], g.cs_f);
  const float w2 = cu.rc2 - gy * gy - gz * gz;
  if (!(w2 >= 0.f)) return false;
  // 1-ulp hardware square root: the cull radius carries a 1e-5 margin
  const float w = __builtin_amdgcn_sqrtf(w2);
  // cells of [x - w, x + w]; the border cells reach to infinity (particles
  // outside the grid are clamped into them), so clamp the range into the grid
  const float last = (float)(g.dims[0] - 1);
  const float fa = fminf(fmaxf(floorf((cu.xd - w) * g.inv_cs_f) - (float)g.lo[0], 0.f), last);
  const float fb = fminf(fmaxf(floorf((cu.xd + w) * g.inv_cs_f) - (float)g.lo[0], 0.f), last);
  int x0 = max(cx - ring, 0), x1 = min(cx + ring, g.dims[0] - 1);
  if (fa > (float)x1 || fb < (float)x0) return false;  // NaN positions keep the ring
  if (fa > (float)x0) x0 = (int)fa;
  if (fb < (float)x1) x1 = (int)fb;
  const int base = (z * g.dims[1] + y) * g.dims[0];
  k0 = base + x0;
  k1 = base + x1 + 1;
  return true;
}

// The particle range [j0, j1) of those cells (empty when there is none).
__device__ __forceinline__ void row_range_cull(const Grid& g, const int* __restrict__ cstart,
                                               int cx, int y, int z, int ring, const Cull& cu,
                                               int& j0, int& j1) {
  j0 = j1 = 0;
  int k0, k1;
  if (!row_cells_cull(g, cx, y, z, ring, cu, k0, k1)) return;
  j0 = cstart[k0];
  j1 = cstart[k1];
}

}  // namespace sph
