// Group scan: 2^k lanes of a wave share one destination particle.
//
// The passes that read the SoA fields (FP64 storage, variable-h symmetric
// pairs, periodic axes, density rates) have few particles more often than
// not, and one lane per destination leaves most of the 1024 SIMDs idle while
// each lane walks its stencil rows one memory latency after another, in
// lanes that wait for the longest row and run the pair arithmetic whenever
// any of the 64 accepts a candidate (per launch, before and with groups:
// FP64 momentum of 60k + 15k particles 400 -> 146 us, of 5k 60 -> 12 us; FP32
// periodic momentum of 100k 1062 -> 197 us).  Here the lanes of a group
//   1. take one stencil row each: cull it to the search sphere, read its two
//      cell starts (one latency for all rows of the group) and append the
//      rows that hold particles to the group's list in LDS;
//   2. take the candidates of the listed rows in turn (lane k of G: the k-th,
//      (k + G)-th, ...), running on from one row into the next, so that every
//      lane gets the same number of candidates whatever the row lengths and
//      the loads of a group are consecutive in memory.
// The caller's step() sees one candidate per lane, in the same order as a
// walk over the rows.  Large sets, whose waves fill the GPU anyway, keep one
// lane per destination (group_log2).
#pragma once
#include "sph_cull.h"

namespace sph {

// k, or the largest smaller number of lanes (log2) with which n destinations
// fit in one launch: a grid holds less than 2^32 threads.
inline int fit_log2(int64_t n, int k) {
  while (k > 0 && (n << k) > (int64_t(1) << 32) - kBlock) --k;
  return k;
}

// Lanes per destination (log2); 0: the plain loops of one lane (for_each_row).
// Eight is the best split from 16k particles on (FP64 momentum of 40k
// particles in 2D: 82 / 68 / 77 us with 4 / 8 / 16 lanes, FP32 periodic in 3D,
// 100k: 231 / 197 / 220 us, FP64 density of 300k: 349 us with 8, 375 with 4);
// smaller sets have too few waves and take 16 (5k: 18.8 / 13.3 / 12.1 us).
// Two sources cull every row twice, which fewer groups per wave make dearer: 4
// lanes once the waves suffice (dam break of 60k + 15k, FP64 momentum: 146 /
// 171 / 213 us; density 66 / 68 / 76).  Once the waves fill the GPU without
// groups, their rows, queues and ballots cost more than they save, sooner in
// 1D and 2D (few rows and pairs a destination) and with two sources, later on
// periodic sets, whose images the groups share out.
// Density + rate + momentum in FP64, 1 (plain loops) / 4 / 8 lanes, in us:
//   1D  20k: 58 / - / 52   50k: 63 / - / 66   100k: 68 / - / 98
//   2D  100k: 218 / 159 / 169   200k: 289 / 275   300k: 374 / 395 / 457
//       1M: 961 / 1257 / 1511   4M: 3438 / 5562 / 6644
//   2D periodic  300k: 519 / 461 / 534   1M (FP32): 922 / 1018 / 1230
//   2D dam break, a step  150k: 415 / 446   300k: 590 / 742   2M: 2416 (8: 4390)
//   3D  300k: 1343 / 1016 / 1034   1M: 3782 / 3364 / 3568   4M: 15877 / 14477 / 15467
//       (clustered 1M: 6365 / 5444 / 5014, so 8 lanes up to there)
inline int group_log2(int64_t n, int nsrc, int dim, bool periodic) {
  if (n < (1 << 14)) return 4;
  if (dim == 1) return n >= (1 << 15) ? 0 : 3;
  const bool few = nsrc >= 2 && n >= (1 << 15);
  if (dim == 3) return fit_log2(n, few || n >= (1 << 20) ? 2 : 3);
  if (n >= (periodic ? 1 << 19 : (nsrc >= 2 ? 1 << 17 : 1 << 18))) return 0;
  return few || n >= (1 << 17) ? 2 : 3;
}

inline int group_blocks(int64_t n, int log2) {
  return (int)((n + (kBlock >> log2) - 1) / (kBlock >> log2));
}

constexpr int kGroupRows = 512;  // row entries per wave, shared by its groups

// LDS of one wave.
struct GroupRows {
  int2 span[kGroupRows];      // [first, last) source slots of a row
  uint8_t image[kGroupRows];  // periodic image code of the row
};

// LDS writes of a wave before, reads after (lanes of one wave run in step).
__device__ __forceinline__ void wave_lds_fence() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// A lane's place in its group.
struct Group {
  int size;    // lanes per destination, a power of two
  int rank;    // this lane's number in the group
  int base;    // first lane of the group
  int index;   // number of the group in the wave
  __device__ __forceinline__ explicit Group(int log2) {
    const int lane = threadIdx.x & 63;
    size = 1 << log2;
    rank = lane & (size - 1);
    base = lane - rank;
    index = lane >> log2;
  }
  // Bits of this group's lanes in a wave mask.
  __device__ __forceinline__ unsigned mine(unsigned long long m) const {
    return (unsigned)(m >> base) & (unsigned)((1ull << size) - 1ull);
  }
  __device__ __forceinline__ int before(unsigned m) const {
    return __popc(m & ((1u << rank) - 1u));
  }
  template <typename V>
  __device__ __forceinline__ V sum(V v) const {
    for (int o = size >> 1; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    return v;
  }
};

// The largest of a block's move bounds (all lanes of all waves) into *disp_out
// by one atomic at most: the atomics go to one address, and one per wave made
// the FP64 stage of 5k particles 24 us instead of 12.
__device__ __forceinline__ void block_raise_max(float* disp_out, float disp) {
  __shared__ float bmax[kBlock / 64];
  for (int o = 32; o > 0; o >>= 1) disp = fmaxf(disp, __shfl_xor(disp, o, 64));
  if ((threadIdx.x & 63) == 0) bmax[threadIdx.x >> 6] = disp;
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int k = 1; k < kBlock / 64; ++k) disp = fmaxf(disp, bmax[k]);
    raise_max(disp_out, disp);
  }
}

// Shift of image code c along the three axes: digits 0, 1, 2 (base 3) stand
// for 0, +1 and -1 periods.
__device__ __forceinline__ double image_shift(int digit, double period) {
  return digit == 0 ? 0.0 : (digit == 1 ? period : -period);
}

// Offset of a periodic image's sources: x_j + s L.
__device__ __forceinline__ double image_offset(int code, int axis, double period) {
  const int d = axis == 0 ? code % 3 : (axis == 1 ? (code / 3) % 3 : code / 9);
  return image_shift(d, period);
}

// Walk every candidate source of the group's destination at (px, py, pz) in
// cell (cx, cy, cz): step(valid, j, image) is called by all lanes of the wave
// together, `valid` lanes with a candidate each.  rc: search radius (any
// displacement since the binning included).  `active` is false for groups
// without a destination.
//
// PERIODIC: the destination's images too, its point shifted by -s L along
// the axes whose face lies within the stencil's reach; sources are then seen
// at x_j + s L, the ghost copy's coordinate (cell.pyx:1277-1376).  Cells of a
// shifted axis come from the image point in FP64 and get one ring more; an
// unshifted axis keeps the destination's own cell.
template <bool PERIODIC, class Step>
__device__ __forceinline__ void group_scan(const Grid& g, const int* __restrict__ cstart,
                                           const Group& gr, GroupRows& L, bool active, double px,
                                           double py, double pz, int cx, int cy, int cz, int ring,
                                           double rc, Step&& step) {
  const int cap = kGroupRows / (64 / gr.size);
  int2* span = L.span + gr.index * cap;
  uint8_t* img = L.image + gr.index * cap;
  int nrows = 0;

  auto candidates = [&]() {
    wave_lds_fence();
    int r = 0, j = 0, j1 = 0, code = 0;
    if (nrows > 0) {
      const int2 s = span[0];
      j = s.x + gr.rank;
      j1 = s.y;
      if (PERIODIC) code = img[0];
    }
    for (;;) {
      // run on into the next rows
      while (r < nrows && j >= j1) {
        ++r;
        if (r < nrows) {
          const int2 s = span[r];
          j = s.x + (j - j1);
          j1 = s.y;
          if (PERIODIC) code = img[r];
        }
      }
      const bool valid = r < nrows;
      if (!__any(valid)) break;
      step(valid, j, code);
      j += gr.size;
    }
    nrows = 0;
    wave_lds_fence();
  };

  // images of this destination: choices per axis (unshifted, lower, upper)
  int nimg = active ? 1 : 0;
  int cnt[3] = {1, 1, 1};
  bool up[3] = {false, false, false};
  if (PERIODIC && active) {
    const double p[3] = {px, py, pz};
    const double reach = ring * g.cs;
#pragma unroll
    for (int a = 0; a < 3; ++a) {
      if (g.per[a] > 0.0) {
        up[a] = p[a] + reach >= g.pmin[a] + g.per[a];
        cnt[a] += (up[a] ? 1 : 0) + (p[a] - reach < g.pmin[a] ? 1 : 0);
      }
    }
    nimg = cnt[0] * cnt[1] * cnt[2];
  }
  for (int im = 0; PERIODIC ? __any(im < nimg) : im == 0; ++im) {
    const bool on = im < nimg;
    double qx = px, qy = py, qz = pz;
    int icx = cx, icy = cy, icz = cz, code = 0, iring = ring;
    if (PERIODIC && im > 0 && on) {
      int d[3] = {im % cnt[0], (im / cnt[0]) % cnt[1], im / (cnt[0] * cnt[1])};
      double q[3] = {px, py, pz};
      int c[3] = {cx, cy, cz};
#pragma unroll
      for (int a = 0; a < 3; ++a) {
        if (d[a] == 1 && !up[a]) d[a] = 2;  // the only shift is the lower one
        if (d[a] != 0) {
          q[a] -= image_shift(d[a], g.per[a]);
          const double k = floor(q[a] / g.cs) - (double)g.lo[a];
          c[a] = !(k >= 0.0) ? 0 : (k > (double)(g.dims[a] - 1) ? g.dims[a] - 1 : (int)k);
        }
      }
      qx = q[0]; qy = q[1]; qz = q[2];
      icx = c[0]; icy = c[1]; icz = c[2];
      code = d[0] + 3 * d[1] + 9 * d[2];
      iring = ring + 1;
    }
    const bool cull = can_cull(g, qx, qy, qz, rc);
    Cull cu{};
    int ylo = max(-iring, -icy), yhi = min(iring, g.dims[1] - 1 - icy);
    int zlo = max(-iring, -icz), zhi = min(iring, g.dims[2] - 1 - icz);
    if (cull) {
      cu = make_cull(make_float4((float)qx, (float)qy, (float)qz, 0.f), rc, g);
      axis_span(cu.yd, cu.r, icy, g.dims[1], g.lo[1], g.inv_cs_f, iring, ylo, yhi);
      axis_span(cu.zd, cu.r, icz, g.dims[2], g.lo[2], g.inv_cs_f, iring, zlo, zhi);
    }
    const int ny = yhi - ylo + 1, nz = zhi - zlo + 1;
    const int total = on && ny > 0 && nz > 0 ? ny * nz : 0;
    // row number q = gr.rank, gr.rank + size, ... as (y, z) offsets
    int y = gr.rank, z = 0;
    for (int q = gr.rank; __any(q - gr.rank < total); q += gr.size) {
      const bool in = q < total;
      while (in && y >= ny) {
        y -= ny;
        ++z;
      }
      int k0 = 0, k1 = 0, j0 = 0, j1 = 0;
      bool row = in;
      if (in) {
        const int ry = icy + ylo + y, rz = icz + zlo + z;
        if (cull) {
          row = row_cells_cull(g, icx, ry, rz, iring, cu, k0, k1);
        } else {
          const int base = (rz * g.dims[1] + ry) * g.dims[0];
          k0 = base + max(icx - iring, 0);
          k1 = base + min(icx + iring, g.dims[0] - 1) + 1;
        }
      }
      if (row) {
        j0 = cstart[k0];
        j1 = cstart[k1];
      }
      const unsigned m = gr.mine(__ballot(j0 < j1));
      if (j0 < j1) {
        const int at = nrows + gr.before(m);
        span[at] = make_int2(j0, j1);
        if (PERIODIC) img[at] = (uint8_t)code;
      }
      nrows += __popc(m);
      y += gr.size;
      if (__any(nrows > cap - gr.size)) candidates();
    }
  }
  candidates();
}

}  // namespace sph
