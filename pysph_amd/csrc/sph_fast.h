// Device building blocks of the packed FP32 neighbour passes, shared by the
// single-array kernels (sph_fast.hip) and the batched multi-scene kernels
// (sph_batch.hip).
//
// Packed FP32 fast path of the neighbour passes.
//
// Inputs are float4 copies per particle: pos4 = (x,y,z,h), vel4 = (u,v,w,m),
// aux4 = (rho,cs,p/rho^2,p) (the FP32 pair arithmetic reads the first three,
// one 12-byte load), optionally pm4 = (x,y,z,m) with the array's h range
// (a density source of uniform h: one load per pair), and the (x,y,z) copy
// pos3 that the candidate screen reads.  One lane per destination particle,
// the particles sorted by cell so that the lanes of a wave share stencil
// rows.
//
// Cell scans: a lane screens the candidates of its stencil rows (four per
// step, three 16-byte loads from pos3) and queues the accepted source
// indices in LDS; when a queue is full, and after each source array, the
// wave drains all queues in one wave-uniform loop, so the pair arithmetic
// runs with ~70% of lanes active instead of the ~40% that accept any one
// candidate.
//
// Neighbour lists: a density scan can record the accepted sources of every
// destination.  Without skin the list holds exactly the neighbours and the
// momentum pass of the same stage reads it without testing again.  With a
// skin the scan records every source within radius*(1+skin) (a superset):
// later passes apply the exact test to each entry, as long as no particle
// has moved more than skin*radius/2 (checked on the device; lanes where it
// fails search the cells again with a widened ring).
//
// Reference formulas: SPHRho (density_funcs.pyx:38-84), TaitEquation
// (eos_funcs.pyx:105-116), MomentumEquation (pressure_funcs.pyx:154-245),
// XSPHCorrection (xsph_funcs.pyx:31-88), cubic spline (kernels.pyx:345-449),
// integrator updates (integrator.py:472-514, :597-619).
#pragma once
#include <math.h>

#include "sph_group.h"
#include "sph_passes.h"

namespace sph {

// LDS queue depth per lane and candidate loads in flight per lane; the
// momentum scans' 24 entries keep six 256-lane blocks within the 160 KiB of
// LDS, the occupancy their 80 VGPRs allow
#ifndef SPH_QUEUE
#define SPH_QUEUE 24
#endif
// LDS queue depth of the density scans (sources of varied h, list builds)
#ifndef SPH_DENS_QUEUE
#define SPH_DENS_QUEUE 16
#endif
#ifndef SPH_UNROLL
#define SPH_UNROLL 4
#endif
constexpr int kQueue = SPH_QUEUE;
constexpr int kDensQueue = SPH_DENS_QUEUE;
// occupancy target of the momentum scan kernels (waves per SIMD)
constexpr int kMomWaves = 6;
constexpr int kUnroll = SPH_UNROLL;
#ifndef SPH_DENS_UNROLL
#define SPH_DENS_UNROLL SPH_UNROLL
#endif
constexpr int kDensUnroll = SPH_DENS_UNROLL;  // candidates per screen step, density
// density sources of uniform h are summed without the LDS queue
#ifndef SPH_DENS_DIRECT
#define SPH_DENS_DIRECT 1
#endif
constexpr bool kDensDirect = SPH_DENS_DIRECT != 0;
// queue-free density sources of uniform mass are read from the (x,y,z) copy
#ifndef SPH_DENS_XYZ
#define SPH_DENS_XYZ 1
#endif
constexpr bool kDensXyz = SPH_DENS_XYZ != 0;
// a density pass over two sources of uniform h sums them row by row
// together (one source, or more than two, take the source-by-source loop)
constexpr int kDirectSrc = 2;
// occupancy target of the density scan kernels (waves per SIMD, 0: none):
// seven waves hold them within 72 VGPRs without spilling
#ifndef SPH_DENS_WAVES
#define SPH_DENS_WAVES 7
#endif
// momentum pairs of a source of uniform h use per-destination constants
#ifndef SPH_MOM_UNI
#define SPH_MOM_UNI 1
#endif
constexpr bool kMomUni = SPH_MOM_UNI != 0;
__device__ constexpr float4 kFar4 = {3.0e38f, 3.0e38f, 3.0e38f, 0.f};

// float4 gather at a non-negative index as a 32-bit byte offset from the
// array base, so the load takes the scalar-base + 32-bit-offset form
// (packed arrays hold at most kPackedMaxN = 2^27 particles).
__device__ __forceinline__ float4 ld4(const float4* __restrict__ base, int j) {
  return *(const float4*)((const char*)base + (unsigned)j * 16u);
}

// compile-time flag for generic lambdas
template <bool B>
struct BoolC {
  static constexpr bool value = B;
};

__device__ __forceinline__ int wave_max(int v) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) v = max(v, __shfl_xor(v, off, 64));
  return v;
}

// Exact neighbour test (FP32 screen, FP64 decision in the band).
__device__ __forceinline__ bool accept_exact(const float4& s, const float4& d, float r2f,
                                             double r2d) {
  const float dx = s.x - d.x, dy = s.y - d.y, dz = s.z - d.z;
  const float d2f = dx * dx + dy * dy + dz * dz;
  return Within32::test(s.x, s.y, s.z, d.x, d.y, d.z, d2f, r2f, r2d);
}

// The pair arithmetic below spells out its fused multiply-adds and forbids
// the compiler others, so that a pair gives the same bits in every kernel it
// is inlined into (the scan of one lane per destination, the groups of lanes
// that share one, the batched scenes).  Sums of products round as
// fma(z, z, fma(x, x, y * y)): the y product alone is rounded, which is how
// the compiler contracts x * x + y * y + z * z by itself.
__device__ __forceinline__ float fma_(float a, float b, float c) { return __builtin_fmaf(a, b, c); }
__device__ __forceinline__ double fma_(double a, double b, double c) {
  return __builtin_fma(a, b, c);
}

template <typename CT>
__device__ __forceinline__ CT pair_d2(const float4& d, const float4& s, CT& rx, CT& ry, CT& rz) {
#pragma clang fp contract(off)
  rx = (CT)d.x - (CT)s.x;
  ry = (CT)d.y - (CT)s.y;
  rz = (CT)d.z - (CT)s.z;
  return fma_(rz, rz, fma_(rx, rx, ry * ry));
}

// Reciprocal and square root: hardware 1-ulp instructions for FP32 pair
// arithmetic, IEEE operations for FP64.
template <typename CT>
__device__ __forceinline__ CT frcp(CT x) {
  return CT(1) / x;
}
template <>
__device__ __forceinline__ float frcp<float>(float x) {
  return __builtin_amdgcn_rcpf(x);
}
template <typename CT>
__device__ __forceinline__ CT fsqrt(CT x) {
  return sqrt(x);
}
template <>
__device__ __forceinline__ float fsqrt<float>(float x) {
  return __builtin_amdgcn_sqrtf(x);
}

// Branch-free cubic spline shape W(q) (kernels.pyx:367-374); t = 2 - q.
template <typename CT>
__device__ __forceinline__ CT w_sel(CT q, CT t) {
#pragma clang fp contract(off)
  const CT outer = CT(0.25) * t * t * t;
  const CT inner = fma_(CT(-1.5) * (q * q), fma_(CT(-0.5), q, CT(1)), CT(1));
  return q > CT(2) ? CT(0) : (q > CT(1) ? outer : inner);
}

template <typename CT>
__device__ __forceinline__ CT w_sel(CT q) {
  return w_sel<CT>(q, CT(2) - q);
}

// Branch-free gradient factor (kernels.pyx:403-412): grad W = r_ab * g.
template <typename CT>
__device__ __forceinline__ CT g_sel(CT q, CT r, CT h, CT inv) {
#pragma clang fp contract(off)
  const CT t = CT(2) - q;
  const CT outer = CT(-0.75) * t * t * frcp<CT>(h * r);
  const CT inner = CT(3) * fma_(CT(0.75), q, CT(-1)) * (inv * inv);
  return q > CT(2) ? CT(0) : (q >= CT(1) ? outer : (q > CT(1e-14) ? inner : CT(0)));
}

// Raw buffer resource over a source's packed positions, the (x,y,z) copy
// when the source has one (n * 12 bytes), else pos4 (n * 16 bytes); gfx9
// resource word 3.  A load at or past the end returns zeros instead of
// touching memory, so candidate loads need no index clamp.
__device__ __forceinline__ __amdgpu_buffer_rsrc_t cand_rsrc(const View<float>& S) {
  if (S.pos3 != nullptr)
    return __builtin_amdgcn_make_buffer_rsrc((void*)S.pos3, (short)0,
                                             (int)((unsigned)S.n * 12u), 0x00020000);
  return __builtin_amdgcn_make_buffer_rsrc((void*)S.pos4, (short)0,
                                           (int)((unsigned)S.n * 16u), 0x00020000);
}

// (x, y, z) of candidate slot u of a block starting at byte offset off.
__device__ __forceinline__ float3 ld_xyz(__amdgpu_buffer_rsrc_t rs, int off) {
  const auto v = __builtin_amdgcn_raw_buffer_load_b96(rs, off, 0, 0);
  return make_float3(__uint_as_float(v[0]), __uint_as_float(v[1]), __uint_as_float(v[2]));
}

// Screen the candidates j0 .. j0+kUnroll-1 (those below j1) of one stencil
// row against destination pd and push the accepted ones into the lane's
// LDS queue q (entries 64 apart), branch-free: every lane loads kUnroll
// candidates through the bounds-checked buffer view `rs` (cand_rsrc: one
// base offset, the slots as immediate offsets, three 16-byte loads per four
// candidates from the (x,y,z) copy, else one 12-byte load each from pos4;
// slots past the row end are loaded but never accepted), writes every
// candidate into the next queue slot and
// advances its count only on acceptance.  The caller keeps
// cnt <= kQueue - kUnroll on entry.  The exact test (Within32) runs its FP64
// branch only when a candidate of some lane falls in the +-2e-6 band; with
// `super` the test is the list-build superset d2 < rl2f instead.
template <int U = kUnroll>
__device__ __forceinline__ void screen_block(const View<float>& S, __amdgpu_buffer_rsrc_t rs,
                                             int j0, int j1, const float4& pd, float r2lo,
                                             float r2hi, double r2d, bool super, float rl2f,
                                             int* q, int& cnt) {
  float3 c[U];
  if (S.pos3 != nullptr && U % 4 == 0) {
    // (x,y,z) copy: four candidates are 48 contiguous bytes, three loads
    int off = (int)((unsigned)j0 * 12u);
    // keep off opaque, so that the slots become immediate load offsets
    // (an empty register constraint: no instruction is emitted)
    asm("" : "+v"(off));
#pragma unroll
    for (int g = 0; g < U / 4; ++g) {
      float w[12];
#pragma unroll
      for (int k = 0; k < 3; ++k) {
        const auto v = __builtin_amdgcn_raw_buffer_load_b128(rs, off + 48 * g + 16 * k, 0, 0);
#pragma unroll
        for (int e = 0; e < 4; ++e) w[4 * k + e] = __uint_as_float(v[e]);
      }
#pragma unroll
      for (int u = 0; u < 4; ++u) c[4 * g + u] = make_float3(w[3 * u], w[3 * u + 1], w[3 * u + 2]);
    }
  } else {
    int off = (int)((unsigned)j0 * 16u);
    asm("" : "+v"(off));
#pragma unroll
    for (int u = 0; u < U; ++u) c[u] = ld_xyz(rs, off + 16 * u);
  }
  const int rem = j1 - j0;
  bool ok[U], bnd[U];
  bool band = false;
#pragma unroll
  for (int u = 0; u < U; ++u) {
    const float dx = c[u].x - pd.x, dy = c[u].y - pd.y, dz = c[u].z - pd.z;
    const float d2f = dx * dx + dy * dy + dz * dz;
    const bool in = u < rem;
    if (super) {
      ok[u] = in && d2f < rl2f;
      bnd[u] = false;
    } else {
      ok[u] = in && d2f < r2lo;
      bnd[u] = in && !(d2f < r2lo) && !(d2f > r2hi);
    }
    band = band || bnd[u];
  }
  if (__any(band)) {
#pragma unroll
    for (int u = 0; u < U; ++u)
      if (bnd[u])
        ok[u] = exact_within((double)c[u].x, (double)c[u].y, (double)c[u].z, (double)pd.x,
                             (double)pd.y, (double)pd.z, r2d);
  }
#pragma unroll
  for (int u = 0; u < U; ++u) {
    q[cnt * 64] = j0 + u;
    cnt += ok[u] ? 1 : 0;
  }
}

// 4^(1/3): with v = 4^(1/3) max(1 - q, 0), v^3 = 4 max(1 - q, 0)^3.
constexpr float kCbrt4 = 1.5874010519681994f;

// 4 w(q) of a pair at squared distance d2, see density_direct_block.
__device__ __forceinline__ float direct_w4(float d2, float ninv, float nkinv) {
  const float s = __builtin_amdgcn_sqrtf(d2);
  // t = max(2 - q, 0) makes w exactly 0 from q = 2 on
  const float t = fmaxf(fmaf(ninv, s, 2.f), 0.f);
  const float v = fmaxf(fmaf(nkinv, s, kCbrt4), 0.f);
  return fmaf(-(v * v), v, t * t * t);
}

// records a wave stages for density_lds_row: its 4 KB LDS region (the
// queue area the queue-free density path does not use)
constexpr int kStage = 256;

// Summation density over U candidate slots of one stencil row of a source
// whose h is uniform: no queue.  `off` is the byte offset of the first slot
// in the source's candidate records, loaded through the bounds-checked
// buffer view `rs` (one base offset, the slots as immediate offsets), and
// `rem` the bytes left in the lane's range, so slot u is a candidate when
// u * stride < rem.  With P3 the records are the 12-byte (x, y, z) copy
// (pos3: four slots in three 16-byte loads, two in a 16-byte and an 8-byte
// load) and every source particle has the mass `mb` (the source's mass is
// uniform); otherwise they are the 16-byte (x, y, z, m) records of pm4.
// Both give the same products, so the same bits; the 12-byte records move a
// quarter fewer bytes through the vector memory pipeline, which the pass
// keeps busy.  With FROM_LDS the records are (x, y, z, m) entries of the
// wave's staged row `stage` (density_lds_row), `off` and `rem` in records
// instead of bytes.  Every lane screens its
// slots like screen_block (FP32 test, FP64 inside the +-2e-6 band) and adds
// m 4w(q) of every accepted one, in row order (the order a queue would
// drain them in).  4w is four times the cubic spline's shape
// (kernels.pyx:367-374), 4 - 6 q^2 + 3 q^3 for q <= 1 and (2 - q)^3 for
// 1 < q < 2, written branch-free as t^3 - v^3 with t = max(2 - q, 0) and
// v = 4^(1/3) max(1 - q, 0) (t^3 - 4 (1 - q)^3 is the inner polynomial),
// q = |r_a - r_b| / h_ab from the screened squared distance; `ninv` =
// -1/h_ab and `nkinv` = -4^(1/3)/h_ab.  The caller scales the row sums by
// fac / 4 (the normalisation of a source of uniform h is the same for every
// pair), which saves the per-pair multiplications by the constants.
// Evaluating w for every slot costs about what queueing the accepted ones
// costs, and it removes the drain loop with its dependent index read,
// gather and memory wait per pair.  FP32 pair arithmetic only.
template <int U, bool P3, bool FROM_LDS = false>
__device__ __forceinline__ void density_direct_block(__amdgpu_buffer_rsrc_t rs, int off, int rem,
                                                     const float4& pd, float r2lo, float r2hi,
                                                     double r2d, float ninv, float nkinv,
                                                     float mb, float& nr,
                                                     const float4* stage = nullptr) {
  static_assert(!P3 || U % 4 == 0 || U == 2, "pos3 blocks: groups of four slots, or two");
  constexpr int kStride = FROM_LDS ? 1 : (P3 ? 12 : 16);
  float4 c[U];
  if constexpr (FROM_LDS) {
#pragma unroll
    for (int u = 0; u < U; ++u) c[u] = stage[(off + u) & (kStage - 1)];
  } else if constexpr (P3 && U == 2) {
    // two slots: 24 bytes, one 16-byte and one 8-byte load
    const auto v = __builtin_amdgcn_raw_buffer_load_b128(rs, off, 0, 0);
    const auto t = __builtin_amdgcn_raw_buffer_load_b64(rs, off + 16, 0, 0);
    c[0] = make_float4(__uint_as_float(v[0]), __uint_as_float(v[1]), __uint_as_float(v[2]), mb);
    c[1] = make_float4(__uint_as_float(v[3]), __uint_as_float(t[0]), __uint_as_float(t[1]), mb);
  } else if constexpr (P3) {
#pragma unroll
    for (int g = 0; g < U / 4; ++g) {
      float w[12];
#pragma unroll
      for (int k = 0; k < 3; ++k) {
        const auto v = __builtin_amdgcn_raw_buffer_load_b128(rs, off + 48 * g + 16 * k, 0, 0);
#pragma unroll
        for (int e = 0; e < 4; ++e) w[4 * k + e] = __uint_as_float(v[e]);
      }
#pragma unroll
      for (int u = 0; u < 4; ++u)
        c[4 * g + u] = make_float4(w[3 * u], w[3 * u + 1], w[3 * u + 2], mb);
    }
  } else {
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const auto v = __builtin_amdgcn_raw_buffer_load_b128(rs, off + 16 * u, 0, 0);
      c[u] = make_float4(__uint_as_float(v[0]), __uint_as_float(v[1]), __uint_as_float(v[2]),
                         __uint_as_float(v[3]));
    }
  }
  bool ok[U], bnd[U];
  float d2[U];
  bool band = false;
#pragma unroll
  for (int u = 0; u < U; ++u) {
    const float dx = c[u].x - pd.x, dy = c[u].y - pd.y, dz = c[u].z - pd.z;
    d2[u] = fmaf(dz, dz, fmaf(dx, dx, dy * dy));
    const bool in = kStride * u < rem;
    const bool lo = d2[u] < r2lo;
    const bool hi = d2[u] <= r2hi;
    ok[u] = in && lo;
    // lo implies hi (r2lo < r2hi); a NaN distance is neither
    bnd[u] = in && (hi != lo);
    band = band || bnd[u];
  }
  if (__any(band)) {
#pragma unroll
    for (int u = 0; u < U; ++u)
      if (bnd[u])
        ok[u] = exact_within((double)c[u].x, (double)c[u].y, (double)c[u].z, (double)pd.x,
                             (double)pd.y, (double)pd.z, r2d);
  }
#pragma unroll
  for (int u = 0; u < U; ++u) nr = fmaf(ok[u] ? c[u].w : 0.f, direct_w4(d2[u], ninv, nkinv), nr);
}

// The candidate records of a density source of uniform h for
// density_direct_block: the (x, y, z) copy when the source also has a
// uniform mass (returned in mb), else the (x, y, z, m) records.
struct DirectSrc {
  __amdgpu_buffer_rsrc_t rs;
  float mb;
  bool p3;
};

__device__ __forceinline__ DirectSrc direct_src(const View<float>& S) {
  DirectSrc d;
  d.p3 = kDensXyz && S.pos3 != nullptr && S.mrange != nullptr && S.mrange[0] == S.mrange[1];
  d.mb = d.p3 ? __int_as_float(S.mrange[0]) : 0.f;
  d.rs = d.p3 ? __builtin_amdgcn_make_buffer_rsrc((void*)S.pos3, (short)0,
                                                  (int)((unsigned)S.n * 12u), 0x00020000)
              : __builtin_amdgcn_make_buffer_rsrc((void*)S.pm4, (short)0,
                                                  (int)((unsigned)S.n * 16u), 0x00020000);
  return d;
}

// Every candidate block of one stencil row [j0, j1) of a direct source.
// From the (x, y, z) copy: blocks of four slots while some lane of the wave
// has four candidates left, then blocks of two, so that fewer slots past
// the lanes' row ends are loaded and screened (the wave runs each block for
// all its lanes; 2^24 cube: 8 % fewer slots).  From the (x, y, z, m)
// records: blocks of four (the second block shape costs that kernel more
// registers than it saves).
__device__ __forceinline__ void density_direct_row(const DirectSrc& d, int j0, int j1,
                                                   const float4& pd, float r2lo, float r2hi,
                                                   double r2d, float inv, float& nr) {
  // byte offsets; off is kept opaque, so that the slots become immediate
  // load offsets (an empty register constraint: no instruction is emitted)
  if (d.p3) {
    int off = (int)((unsigned)j0 * 12u);
    const int end = (int)((unsigned)j1 * 12u);
    asm("" : "+v"(off));
    while (__any(end - off >= 48)) {
      density_direct_block<4, true>(d.rs, off, end - off, pd, r2lo, r2hi, r2d, -inv,
                                    -kCbrt4 * inv, d.mb, nr);
      off += 48;
    }
    while (__any(off < end)) {
      density_direct_block<2, true>(d.rs, off, end - off, pd, r2lo, r2hi, r2d, -inv,
                                    -kCbrt4 * inv, d.mb, nr);
      off += 24;
    }
  } else {
    int off = (int)((unsigned)j0 * 16u);
    const int end = (int)((unsigned)j1 * 16u);
    asm("" : "+v"(off));
    do {
      density_direct_block<4, false>(d.rs, off, end - off, pd, r2lo, r2hi, r2d, -inv,
                                     -kCbrt4 * inv, 0.f, nr);
      off += 64;
    } while (__any(off < end));
  }
}

// Minimum / maximum over the wave (DPP row shifts within rows of 16 lanes,
// then row broadcasts; lane 63 ends with the result).
__device__ __forceinline__ int wave_min_dpp(int v) {
  v = min(v, __builtin_amdgcn_update_dpp(INT_MAX, v, 0x111, 0xf, 0xf, false));
  v = min(v, __builtin_amdgcn_update_dpp(INT_MAX, v, 0x112, 0xf, 0xf, false));
  v = min(v, __builtin_amdgcn_update_dpp(INT_MAX, v, 0x114, 0xf, 0xf, false));
  v = min(v, __builtin_amdgcn_update_dpp(INT_MAX, v, 0x118, 0xf, 0xf, false));
  v = min(v, __builtin_amdgcn_update_dpp(INT_MAX, v, 0x142, 0xa, 0xf, false));
  v = min(v, __builtin_amdgcn_update_dpp(INT_MAX, v, 0x143, 0xc, 0xf, false));
  return __builtin_amdgcn_readlane(v, 63);
}
__device__ __forceinline__ int wave_max_dpp(int v) {
  v = max(v, __builtin_amdgcn_update_dpp(INT_MIN, v, 0x111, 0xf, 0xf, false));
  v = max(v, __builtin_amdgcn_update_dpp(INT_MIN, v, 0x112, 0xf, 0xf, false));
  v = max(v, __builtin_amdgcn_update_dpp(INT_MIN, v, 0x114, 0xf, 0xf, false));
  v = max(v, __builtin_amdgcn_update_dpp(INT_MIN, v, 0x118, 0xf, 0xf, false));
  v = max(v, __builtin_amdgcn_update_dpp(INT_MIN, v, 0x142, 0xa, 0xf, false));
  v = max(v, __builtin_amdgcn_update_dpp(INT_MIN, v, 0x143, 0xc, 0xf, false));
  return __builtin_amdgcn_readlane(v, 63);
}

static_assert(kStage * 16 == kDensQueue * 64 * 4, "one wave's LDS region");

// One stencil row of a direct source through LDS: the wave loads the union
// of its lanes' ranges [lo, hi) of (x, y, z, m) records into its region with
// coalesced 16-byte loads, then every lane screens its own range from LDS
// in the same slot order as density_direct_row (the same sums).  False,
// with nothing done, when the union exceeds the region or a lane's range is
// not inside it.
__device__ __forceinline__ bool density_lds_row(const DirectSrc& d,
                                                const float4* __restrict__ pm4, float4* stage,
                                                int j0, int j1, const float4& pd, float r2lo,
                                                float r2hi, double r2d, float inv, float& nr) {
  const bool has = j0 < j1;
  const int lo = wave_min_dpp(has ? j0 : INT_MAX);
  const int hi = wave_max_dpp(has ? j1 : INT_MIN);
  if (lo >= hi || hi - lo > kStage) return false;
  const int nu = hi - lo;
  if (!__all(!has || (j0 >= lo && j1 <= hi))) return false;
  const int lane = threadIdx.x & 63;
  for (int k = lane; k < nu; k += 64) stage[k] = pm4[lo + k];
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  int o = has ? j0 - lo : 0;
  int rem = has ? j1 - j0 : 0;
  while (__any(rem >= 4)) {
    density_direct_block<4, false, true>(d.rs, o, rem, pd, r2lo, r2hi, r2d, -inv, -kCbrt4 * inv,
                                         0.f, nr, stage);
    o += 4;
    rem -= 4;
  }
  while (__any(rem > 0)) {
    density_direct_block<2, false, true>(d.rs, o, rem, pd, r2lo, r2hi, r2d, -inv, -kCbrt4 * inv,
                                         0.f, nr, stage);
    o += 2;
    rem -= 2;
  }
  // every lane's reads are done before the region is written again
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  return true;
}

// Whether a list built with the given skin still holds every neighbour of a
// destination of search radius r after a displacement of at most disp.
__device__ __forceinline__ bool list_valid(const float* disp, float skin, double r) {
  if (disp == nullptr) return true;
  return 2.0 * (double)(*disp) <= (double)skin * r;
}

// ---------------------------------------------------------------------------
// density
// ---------------------------------------------------------------------------
// W(r_a - r_b, (h_a + h_b) / 2) without fac(1); ps carries the source
// position.
template <typename CT>
__device__ __forceinline__ CT w_value(const float4& pd, const float4& ps, CT hd, CT hb, int dim) {
  CT rx, ry, rz;
  const CT d2 = pair_d2<CT>(pd, ps, rx, ry, rz);
  const CT hab = CT(0.5) * (hd + hb);
  const CT inv = frcp<CT>(hab);
  const CT qq = fsqrt<CT>(d2) * inv;
  return w_sel<CT>(qq) * h_dim_inv<CT>(inv, dim);
}

template <bool TAIT>
__device__ __forceinline__ void density_epilogue(const PassArgs<float>& a, int i, bool local,
                                                 double rho) {
  if (!local) {
    a.rho[i] = 0.f;
    if (TAIT) {
      a.p[i] = 0.f;
      a.cs[i] = 0.f;
    }
    if (a.dst.aux4 != nullptr) a.dst.aux4[i] = make_float4(0.f, 0.f, 0.f, 0.f);
    return;
  }
  const float rhof = (float)rho;
  a.rho[i] = rhof;
  if (TAIT) {
    double p, cs;
    tait((double)rhof, a.co, a.ro, a.gamma, a.B, p, cs);
    const float pf = (float)p;
    a.p[i] = pf;
    a.cs[i] = (float)cs;
    if (a.dst.aux4 != nullptr)
      a.dst.aux4[i] = make_float4(rhof, (float)cs,
                                  (float)((double)pf / ((double)rhof * (double)rhof)), pf);
  }
}

// Cell scan of destination i (all lanes of the wave call it together; q
// is the lane's LDS queue, kDensQueue ints 64 apart); BUILD also records the
// list (superset radius).
// DIM > 0 fixes the dimension at compile time (the kernels of dimensions 2
// and 3); DIM = 0 reads it from the arguments.
template <typename CT, bool TAIT, bool BUILD, int DIM = 0, bool LDS = false>
__device__ __forceinline__ void density_scan_body(const Grid& g, const PassArgs<float>& a,
                                                  int i, int* q) {
#pragma clang fp contract(off)
  const bool valid = i < a.dst.n;
  const bool local = valid && (a.dst.tag == nullptr || a.dst.tag[i] == 0);
  const float4 pd = valid ? a.dst.pos4[i] : make_float4(0.f, 0.f, 0.f, 0.f);
  const double r = (double)pd.w * a.rs;
  const double r2d = r * r;
  const float r2f = (float)r2d;
  // a list built without skin holds exactly the neighbours
  const bool exact_list = !BUILD || a.nl_skin == 0.f;
  const double rl = BUILD ? r * (1.0 + (double)a.nl_skin) : r;
  const float rl2f = (float)(rl * rl) * 1.00001f;
  const float r2lo = r2f * 0.999998f, r2hi = r2f * 1.000002f;
  const bool write_list = BUILD && local;
  int cx = 0, cy = 0, cz = 0;
  if (local) cell_xyz(a.dst.cell[i], g, cx, cy, cz);
  const int ring = ring_of(g, a.disp);
  const double dd = a.disp ? (double)*a.disp : 0.0;
  const Cull cu = make_cull(pd, rl + dd, g);
  int dylo, dyhi, dzlo, dzhi;
  axis_span(cu.yd, cu.r, cy, g.dims[1], g.lo[1], g.inv_cs_f, ring, dylo, dyhi);
  axis_span(cu.zd, cu.r, cz, g.dims[2], g.lo[2], g.inv_cs_f, ring, dzlo, dzhi);
  const int dim = DIM ? DIM : a.dim;
  const CT hd = (CT)pd.w;
  const int64_t ndst = a.dst.n;
  CT rho = CT(0);
  int lpos = 0;
  if constexpr (kDensDirect && !BUILD && sizeof(CT) == 4) {
    // every source of uniform h: the stencil rows outside, the sources
    // inside, so that a row's culled cell range is computed once for all
    // sources; each source keeps its own sum, added in source order (the
    // same bits as summing source by source)
    bool all_uni = a.nsrc >= 2 && a.nsrc <= kDirectSrc;
    for (int s = 0; s < a.nsrc; ++s) {
      const View<float> S = a.src[s];
      all_uni = all_uni && S.pm4 != nullptr && S.hrange != nullptr &&
                S.hrange[0] == S.hrange[1];
    }
    if (all_uni) {
      float inv[kDirectSrc], fac[kDirectSrc], nrs[kDirectSrc];
      bool scan[kDirectSrc];
      DirectSrc ds[kDirectSrc];
#pragma unroll
      for (int s = 0; s < kDirectSrc; ++s) {
        ds[s] = direct_src(a.src[s < a.nsrc ? s : 0]);
        nrs[s] = 0.f;
        scan[s] = s < a.nsrc && !(s == a.cache_src && a.cache_mode == 2);
        const float hb = s < a.nsrc ? __int_as_float(a.src[s].hrange[0]) : 1.f;
        const float hab = 0.5f * ((float)hd + hb);
        inv[s] = frcp<float>(hab);
        fac[s] = h_dim_inv<float>(inv[s], dim);
      }
      for (int dz = -ring; dz <= ring; ++dz) {
        const bool zok = local && dz >= dzlo && dz <= dzhi;
        if (!__any(zok)) continue;
        for (int dy = -ring; dy <= ring; ++dy) {
          const bool yok = zok && dy >= dylo && dy <= dyhi;
          if (!__any(yok)) continue;
          int k0 = 0, k1 = 0;
          const bool row = yok && row_cells_cull(g, cx, cy + dy, cz + dz, ring, cu, k0, k1);
#pragma unroll
          for (int s = 0; s < kDirectSrc; ++s) {
            if (!scan[s]) continue;
            const View<float> S = a.src[s];
            int j0 = 0, j1 = 0;
            if (row) {
              j0 = S.cstart[k0];
              j1 = S.cstart[k1];
            }
            if (!__any(j0 < j1)) continue;
            if (!(LDS && density_lds_row(ds[s], S.pm4, (float4*)(q - (threadIdx.x & 63)), j0,
                                         j1, pd, r2lo, r2hi, r2d, inv[s], nrs[s])))
              density_direct_row(ds[s], j0, j1, pd, r2lo, r2hi, r2d, inv[s], nrs[s]);
          }
        }
      }
#pragma unroll
      for (int s = 0; s < kDirectSrc; ++s) {
        if (s >= a.nsrc) continue;
        CT nr = (CT)(nrs[s] * (0.25f * fac[s]));
        if (s == a.cache_src && a.cache_mode == 2) {
          if (local) nr = (CT)a.cache_sums[i];
        } else if (s == a.cache_src && a.cache_mode == 1 && valid) {
          a.cache_sums[i] = (double)nr;
        }
        rho += nr;
      }
      if (!valid) return;
      density_epilogue<TAIT>(a, i, local, (double)(rho * (CT)a.fac1));
      return;
    }
  }
  for (int s = 0; s < a.nsrc; ++s) {
    const View<float> S = a.src[s];
    const __amdgpu_buffer_rsrc_t rs = cand_rsrc(S);
    CT nr = CT(0);
    if (!BUILD && s == a.cache_src && a.cache_mode == 2) {
      // stored partial sum of a static source (exact round trip via double)
      if (local) nr = (CT)a.cache_sums[i];
      rho += nr;
      continue;
    }
    int cnt = 0, cnt_s = 0;
    // a source of uniform h with an (x,y,z,m) copy: one 16-byte record per
    // pair, h_b from the source's h-uniformity pair (the same value, the
    // same bits)
    const bool uni_h = exact_list && S.pm4 != nullptr && S.hrange != nullptr &&
                       S.hrange[0] == S.hrange[1];
    const CT h_src = uni_h ? (CT)__int_as_float(S.hrange[0]) : CT(0);
    if (kDensDirect && !BUILD && uni_h && sizeof(CT) == 4) {
      // queue-free summation (density_direct_block): h_ab, 1/h_ab and the
      // kernel normalisation are fixed per destination and source
      const float hab = 0.5f * ((float)hd + (float)h_src);
      const float inv = frcp<float>(hab);
      const float fac = h_dim_inv<float>(inv, dim);
      float nrf = 0.f;
      const DirectSrc d = direct_src(S);
      for (int dz = -ring; dz <= ring; ++dz) {
        const bool zok = local && dz >= dzlo && dz <= dzhi;
        if (!__any(zok)) continue;
        for (int dy = -ring; dy <= ring; ++dy) {
          const bool yok = zok && dy >= dylo && dy <= dyhi;
          if (!__any(yok)) continue;
          int j0 = 0, j1 = 0;
          if (yok) row_range_cull(g, S.cstart, cx, cy + dy, cz + dz, ring, cu, j0, j1);
          if (__any(j0 < j1)) {
            if (!(LDS && density_lds_row(d, S.pm4, (float4*)(q - (threadIdx.x & 63)), j0, j1,
                                         pd, r2lo, r2hi, r2d, inv, nrf)))
              density_direct_row(d, j0, j1, pd, r2lo, r2hi, r2d, inv, nrf);
          }
        }
      }
      nr = (CT)(nrf * (0.25f * fac));
      if (s == a.cache_src && a.cache_mode == 1 && valid) a.cache_sums[i] = (double)nr;
      rho += nr;
      continue;
    }
    auto drain = [&]() {
      if (uni_h) {
        for (int k = 0; __any(k < cnt); ++k) {
          if (k < cnt) {
            const int j = q[k * 64];
            const float4 pm = ld4(S.pm4, j);
            nr = fma_((CT)pm.w, w_value<CT>(pd, pm, hd, h_src, dim), nr);
            if (write_list && lpos + k < a.nl_max) a.nl_idx[(int64_t)(lpos + k) * ndst + i] = j;
          }
        }
      } else {
        for (int k = 0; __any(k < cnt); ++k) {
          if (k < cnt) {
            const int j = q[k * 64];
            const float4 ps = ld4(S.pos4, j);
            if (exact_list || accept_exact(ps, pd, r2f, r2d))
              nr = fma_((CT)ld4(S.vel4, j).w, w_value<CT>(pd, ps, hd, (CT)ps.w, dim), nr);
            if (write_list && lpos + k < a.nl_max) a.nl_idx[(int64_t)(lpos + k) * ndst + i] = j;
          }
        }
      }
      lpos += cnt;
      cnt_s += cnt;
      cnt = 0;
    };
    for (int dz = -ring; dz <= ring; ++dz) {
      const bool zok = local && dz >= dzlo && dz <= dzhi;
      if (!__any(zok)) continue;
      for (int dy = -ring; dy <= ring; ++dy) {
        const bool yok = zok && dy >= dylo && dy <= dyhi;
        if (!__any(yok)) continue;
        int j0 = 0, j1 = 0;
        if (yok) row_range_cull(g, S.cstart, cx, cy + dy, cz + dz, ring, cu, j0, j1);
        while (__any(j0 < j1)) {
          if (__any(cnt > kDensQueue - kDensUnroll)) drain();
          screen_block<kDensUnroll>(S, rs, j0, j1, pd, r2lo, r2hi, r2d, !exact_list, rl2f, q,
                                    cnt);
          j0 += kDensUnroll;
        }
      }
    }
    drain();
    if (!BUILD && s == a.cache_src && a.cache_mode == 1 && valid) a.cache_sums[i] = (double)nr;
    rho += nr;
    if (BUILD && valid) a.nl_count[(int64_t)s * ndst + i] = local ? cnt_s : 0;
  }
  if (!valid) return;
  density_epilogue<TAIT>(a, i, local, (double)(rho * (CT)a.fac1));
}
// ---------------------------------------------------------------------------
// momentum + XSPH (+ integrator update)
// ---------------------------------------------------------------------------
template <typename CT>
struct MomDst {
  CT ha, rhoa, ca, Aa, alpha, beta, eta2;
  float4 pd, vd;
  int dim;
};

// What a pair adds to the sums of its destination: gf * (rx, ry, rz) to the
// momentum sum, temp * -(vx, vy, vz) to the XSPH sum (v_b - v_a = -(v_a - v_b)
// exactly).
template <typename CT>
struct PairTerms {
  CT gf, rx, ry, rz, temp, vx, vy, vz;
};

template <typename CT, bool DM, bool DX>
__device__ __forceinline__ void mom_add(const PairTerms<CT>& t, CT* am, CT* ax) {
  if (DM) {
    am[0] = fma_(t.gf, t.rx, am[0]);
    am[1] = fma_(t.gf, t.ry, am[1]);
    am[2] = fma_(t.gf, t.rz, am[2]);
  }
  if (DX) {
    ax[0] = fma_(t.temp, -t.vx, ax[0]);
    ax[1] = fma_(t.temp, -t.vy, ax[1]);
    ax[2] = fma_(t.temp, -t.vz, ax[2]);
  }
}

// One pair of the momentum (DM) and XSPH (DX) sums.  The roles are fixed
// at compile time, so no branch separates a pair's gathers: the compiler
// would otherwise sink the loads that only one role uses behind that
// role's branch, and wait for memory twice per pair.
template <typename CT, bool DM, bool DX>
__device__ __forceinline__ PairTerms<CT> mom_terms_r(const MomDst<CT>& D, const float4& ps,
                                                     const float4& vs, const float4& as) {
#pragma clang fp contract(off)
  PairTerms<CT> T{};
  const CT d2 = pair_d2<CT>(D.pd, ps, T.rx, T.ry, T.rz);
  const CT hab = CT(0.5) * (D.ha + (CT)ps.w);
  const CT inv = frcp<CT>(hab);
  const CT rr = fsqrt<CT>(d2);
  const CT qq = rr * inv;
  const CT fac = h_dim_inv<CT>(inv, D.dim);
  const CT mb = (CT)vs.w;
  const CT rhob = (CT)as.x;
  const CT irhoab = frcp<CT>(CT(0.5) * (D.rhoa + rhob));
  // every source field is read before the branches, so the three gathers of
  // a pair go out together
  T.vx = (CT)D.vd.x - (CT)vs.x;
  T.vy = (CT)D.vd.y - (CT)vs.y;
  T.vz = (CT)D.vd.z - (CT)vs.z;
  const CT Ab = sizeof(CT) == 8 ? (CT)as.w / (rhob * rhob) : (CT)as.z;
  const CT cab = CT(0.5) * (D.ca + (CT)as.y);
  if (DM) {
    const CT dot = fma_(T.vz, T.rz, fma_(T.vx, T.rx, T.vy * T.ry));
    const CT mu = hab * dot * frcp<CT>(fma_(D.eta2 * hab, hab, d2));
    const CT piab = fma_(D.beta * mu, mu, -D.alpha * cab * mu) * irhoab;
    const CT tmp = D.Aa + Ab + (dot < CT(0) ? piab : CT(0));
    T.gf = -mb * tmp * (g_sel<CT>(qq, rr, hab, inv) * fac);
  }
  if (DX) T.temp = mb * (w_sel<CT>(qq) * fac) * irhoab;
  return T;
}

// Constants of the pairs of one destination with a source whose h is
// uniform (h_b fixed): h_ab, 1/h_ab, the normalisation 1/h_ab^dim and the
// gradient factors folded with it.
struct MomUni {
  float hab, inv, fac, eta2hh, kout, kin;
};

__device__ __forceinline__ MomUni mom_uni(float ha, float hb, float eta2, int dim) {
  MomUni u;
  u.hab = 0.5f * (ha + hb);
  u.inv = frcp<float>(u.hab);
  u.fac = h_dim_inv<float>(u.inv, dim);
  u.eta2hh = eta2 * u.hab * u.hab;
  u.kout = -0.75f * u.inv * u.fac;
  u.kin = 3.0f * (u.inv * u.inv) * u.fac;
  return u;
}

// mom_terms_r<float, DM, DX> for a source of uniform h: the per-pair
// reciprocal of h_ab and the normalisation come from MomUni, and one
// reciprocal square root gives both |r_ab| and the 1/|r_ab| of the outer
// gradient branch (kernels.pyx:403-412), so a pair costs three
// quarter-rate transcendental instructions instead of five.
template <bool DM, bool DX>
__device__ __forceinline__ PairTerms<float> mom_terms_u(const MomDst<float>& D, const MomUni& U,
                                                        const float4& ps, const float4& vs,
                                                        const float4& as) {
#pragma clang fp contract(off)
  PairTerms<float> T{};
  const float d2 = pair_d2<float>(D.pd, ps, T.rx, T.ry, T.rz);
  const float rs = __builtin_amdgcn_rsqf(d2);
  const float rr = d2 > 0.f ? d2 * rs : 0.f;  // the self pair: r = 0, not 0 * inf
  const float qq = rr * U.inv;
  // 2 - r / h_ab: one rounding where both sums share it
  const float t = DM && DX ? fma_(-U.inv, rr, 2.f) : 2.f - qq;
  const float mb = vs.w;
  const float rhob = as.x;
  const float irhoab = frcp<float>(0.5f * (D.rhoa + rhob));
  T.vx = D.vd.x - vs.x;
  T.vy = D.vd.y - vs.y;
  T.vz = D.vd.z - vs.z;
  const float Ab = as.z;
  const float cab = 0.5f * (D.ca + as.y);
  if (DM) {
    const float dot = fma_(T.vz, T.rz, fma_(T.vx, T.rx, T.vy * T.ry));
    const float mu = U.hab * dot * frcp<float>(d2 + U.eta2hh);
    const float piab = fma_(D.beta * mu, mu, -D.alpha * cab * mu) * irhoab;
    const float tmp = D.Aa + Ab + (dot < 0.f ? piab : 0.f);
    const float outer = U.kout * (t * t) * rs;
    const float inner = U.kin * fma_(0.75f, qq, -1.f);
    const float gfac = qq > 2.f ? 0.f : (qq >= 1.f ? outer : (qq > 1e-14f ? inner : 0.f));
    T.gf = -mb * tmp * gfac;
  }
  if (DX) T.temp = mb * (w_sel<float>(qq, t) * U.fac) * irhoab;
  return T;
}

// The same pair with the roles chosen at run time (list passes).
template <typename CT>
__device__ __forceinline__ void mom_pair(const MomDst<CT>& D, const float4& ps, const float4& vs,
                                         const float4& as, bool do_m, bool do_x, CT* am,
                                         CT* ax) {
  if (do_m && do_x)
    mom_add<CT, true, true>(mom_terms_r<CT, true, true>(D, ps, vs, as), am, ax);
  else if (do_m)
    mom_add<CT, true, false>(mom_terms_r<CT, true, false>(D, ps, vs, as), am, ax);
  else if (do_x)
    mom_add<CT, false, true>(mom_terms_r<CT, false, true>(D, ps, vs, as), am, ax);
}

template <typename CT, int DIM = 0>
__device__ __forceinline__ MomDst<CT> mom_dst(const PassArgs<float>& a, int i, bool valid) {
  const float4 zero4 = make_float4(0.f, 0.f, 0.f, 0.f);
  MomDst<CT> D;
  D.pd = valid ? a.dst.pos4[i] : zero4;
  D.vd = valid ? a.dst.vel4[i] : zero4;
  const float4 ad = valid ? a.dst.aux4[i] : zero4;
  D.dim = DIM ? DIM : a.dim;
  D.ha = (CT)D.pd.w;
  D.rhoa = (CT)ad.x;
  D.ca = (CT)ad.y;
  D.Aa = sizeof(CT) == 8 ? (CT)ad.w / (D.rhoa * D.rhoa) : (CT)ad.z;
  D.alpha = (CT)a.alpha;
  D.beta = (CT)a.beta;
  D.eta2 = (CT)(a.eta * a.eta);
  return D;
}

// Outputs of the plain pass (MODE 0) or the integrator update of one
// particle in the reference's per-calc order mom, gravity, step, xsph
// (MODE 1 RK2 predictor, 2 RK2 final, 3 Euler); see momentum_kernel.
// Returns the bound of the particle's move (modes 1 to 3; 0 for mode 0).
template <typename CT, int MODE>
__device__ __forceinline__ float mom_epilogue(const PassArgs<float>& a, int i, bool local,
                                              CT* acc, CT* dv, const float4& vd) {
#pragma clang fp contract(off)
  const CT f1 = (CT)a.fac1, fe = (CT)(a.fac1 * a.eps);
#pragma unroll
  for (int c = 0; c < 3; ++c) {
    acc[c] *= f1;
    dv[c] *= fe;
  }
  if (MODE == 0) {
    for (int c = 0; c < 3; ++c) {
      if (a.do_mom && a.acc[c] != nullptr) a.acc[c][i] = (float)acc[c];
      if (a.do_xsph && a.dv[c] != nullptr) a.dv[c][i] = (float)dv[c];
    }
    return 0.f;
  }
  const float dt = (float)a.dt;
  const float hdt = (float)(0.5 * a.dt);
  const float vel[3] = {vd.x, vd.y, vd.z};
  double mv2 = 0.0;
  for (int c = 0; c < a.dim; ++c) {
    const float x0 = a.s0[c][i];
    const float u0 = a.s0[3 + c][i];
    const float km = local ? (float)acc[c] : 0.f;
    const float kx = local ? (float)dv[c] : 0.f;
    const float kg = (local && a.has_gravity) ? (float)a.g[c] : 0.f;
    const float ks = local ? vel[c] : 0.f;
    float xn, un;
    if (MODE == 1 || MODE == 3) {
      un = fma_(km, dt, u0);
      if (a.has_gravity) un = fma_(kg, dt, un);
      xn = fma_(ks, dt, x0);
      if (a.do_xsph) xn = fma_(kx, dt, xn);
      if (MODE == 1) {
        a.k1[c][i] = km;
        a.k1[3 + c][i] = kx;
      }
    } else {
      const float k1m = a.k1[c][i], k1x = a.k1[3 + c][i];
      un = fma_(hdt, k1m + km, u0);
      if (a.has_gravity) un = fma_(hdt, kg + kg, un);
      xn = fma_(hdt, u0 + ks, x0);
      if (a.do_xsph) xn = fma_(hdt, k1x + kx, xn);
    }
    a.out[c][i] = xn;
    a.out[3 + c][i] = un;
    const double mv = (double)xn - (double)x0;  // exact for two floats this close
    mv2 += mv * mv;
  }
  return move_bound(mv2);
}

// The largest of a wave's move bounds into *disp_out.
__device__ __forceinline__ void wave_raise_max(float* disp_out, float disp) {
  for (int off = 32; off > 0; off >>= 1) disp = fmaxf(disp, __shfl_xor(disp, off, 64));
  if ((threadIdx.x & 63) == 0) raise_max(disp_out, disp);
}

// Cell scan with LDS queues (no list) for destination i; q as in
// density_scan_body.
template <typename CT, int MODE, int DIM = 0>
__device__ __forceinline__ void momentum_scan_body(const Grid& g, const PassArgs<float>& a,
                                                   int i, int* q) {
  const bool valid = i < a.dst.n;
  const bool local = valid && (a.dst.tag == nullptr || a.dst.tag[i] == 0);
  const MomDst<CT> D = mom_dst<CT, DIM>(a, i, valid);
  const double r = (double)D.pd.w * a.rs;
  const double r2d = r * r;
  const float r2f = (float)r2d;
  const float r2lo = r2f * 0.999998f, r2hi = r2f * 1.000002f;
  int cx = 0, cy = 0, cz = 0;
  if (local) cell_xyz(a.dst.cell[i], g, cx, cy, cz);
  const int ring = ring_of(g, a.disp);
  const Cull cu = make_cull(D.pd, r + (a.disp ? (double)*a.disp : 0.0), g);
  int dylo, dyhi, dzlo, dzhi;
  axis_span(cu.yd, cu.r, cy, g.dims[1], g.lo[1], g.inv_cs_f, ring, dylo, dyhi);
  axis_span(cu.zd, cu.r, cz, g.dims[2], g.lo[2], g.inv_cs_f, ring, dzlo, dzhi);
  CT acc[3] = {CT(0), CT(0), CT(0)};
  CT dv[3] = {CT(0), CT(0), CT(0)};
  for (int s = 0; s < a.nsrc; ++s) {
    const View<float> S = a.src[s];
    const __amdgpu_buffer_rsrc_t rs = cand_rsrc(S);
    const bool do_m = (a.flags[s] & SPH_SRC_MOMENTUM) != 0 && a.do_mom;
    const bool do_x = (a.flags[s] & SPH_SRC_XSPH) != 0 && a.do_xsph;
    if (!do_m && !do_x) continue;
    CT am[3] = {CT(0), CT(0), CT(0)};
    CT ax[3] = {CT(0), CT(0), CT(0)};
    int cnt = 0;
    // a source of uniform h (FP32 pairs): per-destination pair constants
    const bool uni = kMomUni && sizeof(CT) == 4 && S.hrange != nullptr &&
                     S.hrange[0] == S.hrange[1];
    // one drain loop per role set (the roles are uniform over a source)
    auto drain_r = [&](auto dm, auto dx) {
      constexpr bool M = decltype(dm)::value, X = decltype(dx)::value;
      if constexpr (sizeof(CT) == 4) {
        if (uni) {
          // formed per drain, so that they hold no registers while screening
          const MomUni U = mom_uni((float)D.ha, __int_as_float(S.hrange[0]), (float)D.eta2,
                                   D.dim);
          for (int k = 0; __any(k < cnt); ++k) {
            if (k < cnt) {
              const int j = q[k * 64];
              mom_add<float, M, X>(
                  mom_terms_u<M, X>(reinterpret_cast<const MomDst<float>&>(D), U, ld4(S.pos4, j),
                                    ld4(S.vel4, j), ld4(S.aux4, j)),
                  (float*)am, (float*)ax);
            }
          }
          cnt = 0;
          return;
        }
      }
      for (int k = 0; __any(k < cnt); ++k) {
        if (k < cnt) {
          const int j = q[k * 64];
          mom_add<CT, M, X>(
              mom_terms_r<CT, M, X>(D, ld4(S.pos4, j), ld4(S.vel4, j), ld4(S.aux4, j)), am, ax);
        }
      }
      cnt = 0;
    };
    auto drain = [&]() {
      if (do_m && do_x)
        drain_r(BoolC<true>{}, BoolC<true>{});
      else if (do_m)
        drain_r(BoolC<true>{}, BoolC<false>{});
      else
        drain_r(BoolC<false>{}, BoolC<true>{});
    };
    for (int dz = -ring; dz <= ring; ++dz) {
      const bool zok = local && dz >= dzlo && dz <= dzhi;
      if (!__any(zok)) continue;
      for (int dy = -ring; dy <= ring; ++dy) {
        const bool yok = zok && dy >= dylo && dy <= dyhi;
        if (!__any(yok)) continue;
        int j0 = 0, j1 = 0;
        if (yok) row_range_cull(g, S.cstart, cx, cy + dy, cz + dz, ring, cu, j0, j1);
        while (__any(j0 < j1)) {
          if (__any(cnt > kQueue - kUnroll)) drain();
          screen_block(S, rs, j0, j1, D.pd, r2lo, r2hi, r2d, false, 0.f, q, cnt);
          j0 += kUnroll;
        }
      }
    }
    drain();
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      acc[c] += am[c];
      dv[c] += ax[c];
    }
  }
  if (!valid) return;
  const float disp = mom_epilogue<CT, MODE>(a, i, local, acc, dv, D.vd);
  if (MODE != 0 && a.disp_out != nullptr) wave_raise_max(a.disp_out, disp);
}

// ---------------------------------------------------------------------------
// groups of lanes sharing a destination (sph_group.h), packed FP32 inputs
// ---------------------------------------------------------------------------
// Small sets leave most SIMDs idle at one lane per destination, and each
// lane then pays its rows' and pairs' latencies one after another (2D dam
// break of 1.5k + 0.8k particles: density 18, stage 31 us a launch; with 16
// lanes 12 and 12; the lines are at small_log2).  The
// groups below give the same bits as the scans above: they visit the same
// accepted sources in the same order, each lane works out the terms of one
// pair (the arithmetic spells out its roundings), and the terms are added
// one after another in that order, a sum per lane of the group.
constexpr int kSmallQueue = 1024;  // queued sources per wave, shared by its groups
constexpr int kTermPitch = 9;      // floats per lane: the groups of a wave use other banks

struct SmallLds {
  GroupRows rows;
  int queue[kSmallQueue];
  float terms[64 * kTermPitch];
};

// Ordered accepted sources of S: drain(queue, count) is called with the
// group's queue, in pieces, by all lanes of the wave.
template <class Drain>
__device__ __forceinline__ void small_scan(const Grid& g, const View<float>& S, const Group& gr,
                                           SmallLds& L, bool local, const float4& pd, int cx,
                                           int cy, int cz, int ring, double rc, float r2lo,
                                           float r2hi, double r2d, Drain&& drain) {
  const int cap = kSmallQueue / (64 / gr.size);
  int* q = L.queue + gr.index * cap;
  int count = 0;
  auto empty = [&]() {
    wave_lds_fence();
    drain(q, count);
    count = 0;
    wave_lds_fence();
  };
  group_scan<false>(g, S.cstart, gr, L.rows, local, (double)pd.x, (double)pd.y, (double)pd.z, cx,
                    cy, cz, ring, rc, [&](bool valid, int j, int) {
    bool ok = false;
    if (valid) {
      float x, y, z;
      if (S.pos3 != nullptr) {
        const float* c = S.pos3 + 3 * (int64_t)j;
        x = c[0];
        y = c[1];
        z = c[2];
      } else {
        const float4 c = ld4(S.pos4, j);
        x = c.x;
        y = c.y;
        z = c.z;
      }
      const float dx = x - pd.x, dy = y - pd.y, dz = z - pd.z;
      const float d2f = dx * dx + dy * dy + dz * dz;
      ok = d2f < r2lo;
      if (!ok && d2f <= r2hi)
        ok = exact_within((double)x, (double)y, (double)z, (double)pd.x, (double)pd.y,
                          (double)pd.z, r2d);
    }
    const unsigned m = gr.mine(__ballot(ok));
    if (ok) q[count + gr.before(m)] = j;
    count += __popc(m);
    if (__any(count > cap - gr.size)) empty();
  });
  empty();
}

// density_scan_body<float> (no list, no source cache) for the group of
// destination i.
template <bool TAIT, int DIM>
__device__ __forceinline__ void density_small_body(const Grid& g, const PassArgs<float>& a,
                                                   const Group& gr, int i, SmallLds& L) {
#pragma clang fp contract(off)
  const bool valid = i < a.dst.n;
  const bool local = valid && (a.dst.tag == nullptr || a.dst.tag[i] == 0);
  const float4 pd = valid ? a.dst.pos4[i] : make_float4(0.f, 0.f, 0.f, 0.f);
  const double r = (double)pd.w * a.rs;
  const double r2d = r * r;
  const float r2f = (float)r2d;
  const float r2lo = r2f * 0.999998f, r2hi = r2f * 1.000002f;
  int cx = 0, cy = 0, cz = 0;
  if (local) cell_xyz(a.dst.cell[i], g, cx, cy, cz);
  const int ring = ring_of(g, a.disp);
  const double rc = r + (a.disp ? (double)*a.disp : 0.0);
  const int dim = DIM ? DIM : a.dim;
  float* terms = L.terms + gr.base * kTermPitch;
  float rho = 0.f;
  for (int s = 0; s < a.nsrc; ++s) {
    const View<float> S = a.src[s];
    const bool uni = kDensDirect && S.pm4 != nullptr && S.hrange != nullptr &&
                     S.hrange[0] == S.hrange[1];
    const float hb = uni ? __int_as_float(S.hrange[0]) : 1.f;
    const float inv = frcp<float>(0.5f * (pd.w + hb));
    const float fac = h_dim_inv<float>(inv, dim);
    float nr = 0.f;
    small_scan(g, S, gr, L, local, pd, cx, cy, cz, ring, rc, r2lo, r2hi, r2d,
               [&](const int* q, int count) {
      for (int b = 0; __any(b < count); b += gr.size) {
        const int k = b + gr.rank;
        float m = 0.f, w = 0.f;
        if (k < count) {
          const int j = q[k];
          if (uni) {
            const float4 c = ld4(S.pm4, j);
            const float dx = c.x - pd.x, dy = c.y - pd.y, dz = c.z - pd.z;
            const float d2 = fmaf(dz, dz, fmaf(dx, dx, dy * dy));
            m = c.w;
            w = direct_w4(d2, -inv, -kCbrt4 * inv);
          } else {
            const float4 c = ld4(S.pos4, j);
            m = ld4(S.vel4, j).w;
            w = w_value<float>(pd, c, pd.w, c.w, dim);
          }
        }
        terms[gr.rank * kTermPitch] = m;
        terms[gr.rank * kTermPitch + 1] = w;
        wave_lds_fence();
        // lanes without a pair left zeros, which add nothing
        if (gr.rank == 0) {
          for (int t0 = 0; t0 < gr.size; t0 += 8)
#pragma unroll
            for (int t = 0; t < 8; ++t)
              nr = fmaf(terms[(t0 + t) * kTermPitch], terms[(t0 + t) * kTermPitch + 1], nr);
        }
        wave_lds_fence();
      }
    });
    rho += uni ? nr * (0.25f * fac) : nr;
  }
  if (!valid || gr.rank != 0) return;
  density_epilogue<TAIT>(a, i, local, (double)(rho * (float)a.fac1));
}

// momentum_scan_body<float, MODE> for the group of destination i (groups of
// at least eight lanes: one sum component per lane).
template <int MODE, int DIM>
__device__ __forceinline__ void momentum_small_body(const Grid& g, const PassArgs<float>& a,
                                                    const Group& gr, int i, SmallLds& L) {
  const bool valid = i < a.dst.n;
  const bool local = valid && (a.dst.tag == nullptr || a.dst.tag[i] == 0);
  const MomDst<float> D = mom_dst<float, DIM>(a, i, valid);
  const double r = (double)D.pd.w * a.rs;
  const double r2d = r * r;
  const float r2f = (float)r2d;
  const float r2lo = r2f * 0.999998f, r2hi = r2f * 1.000002f;
  int cx = 0, cy = 0, cz = 0;
  if (local) cell_xyz(a.dst.cell[i], g, cx, cy, cz);
  const int ring = ring_of(g, a.disp);
  const double rc = r + (a.disp ? (double)*a.disp : 0.0);
  float* terms = L.terms + gr.base * kTermPitch;
  // lane c of the group holds component c of (momentum, XSPH)
  const int comp = gr.rank;
  const float sign = comp < 3 ? 1.f : -1.f;
  const int fa = comp < 3 ? 0 : 4, fb = comp < 3 ? 1 + comp : 2 + comp;
  float total = 0.f;
  for (int s = 0; s < a.nsrc; ++s) {
    const View<float> S = a.src[s];
    const bool do_m = (a.flags[s] & SPH_SRC_MOMENTUM) != 0 && a.do_mom;
    const bool do_x = (a.flags[s] & SPH_SRC_XSPH) != 0 && a.do_xsph;
    if (!do_m && !do_x) continue;
    const bool uni = kMomUni && S.hrange != nullptr && S.hrange[0] == S.hrange[1];
    const MomUni U = mom_uni(D.ha, uni ? __int_as_float(S.hrange[0]) : 1.f, D.eta2, D.dim);
    const bool mine = comp < 6 && (comp < 3 ? do_m : do_x);
    float sum = 0.f;
    small_scan(g, S, gr, L, local, D.pd, cx, cy, cz, ring, rc, r2lo, r2hi, r2d,
               [&](const int* q, int count) {
      for (int b = 0; __any(b < count); b += gr.size) {
        const int k = b + gr.rank;
        PairTerms<float> T{};
        if (k < count) {
          const int j = q[k];
          const float4 ps = ld4(S.pos4, j), vs = ld4(S.vel4, j), as = ld4(S.aux4, j);
          // a source's roles are part of a pair's rounding (mom_terms_u)
          if (!uni)
            T = mom_terms_r<float, true, true>(D, ps, vs, as);
          else if (do_m && do_x)
            T = mom_terms_u<true, true>(D, U, ps, vs, as);
          else if (do_m)
            T = mom_terms_u<true, false>(D, U, ps, vs, as);
          else
            T = mom_terms_u<false, true>(D, U, ps, vs, as);
        }
        float* tp = terms + gr.rank * kTermPitch;
        tp[0] = T.gf;
        tp[1] = T.rx;
        tp[2] = T.ry;
        tp[3] = T.rz;
        tp[4] = T.temp;
        tp[5] = T.vx;
        tp[6] = T.vy;
        tp[7] = T.vz;
        wave_lds_fence();
        // lanes without a pair left zeros, which add nothing
        if (mine) {
          for (int t0 = 0; t0 < gr.size; t0 += 8)
#pragma unroll
            for (int t = 0; t < 8; ++t) {
              const float* p = terms + (t0 + t) * kTermPitch;
              sum = fmaf(p[fa], sign * p[fb], sum);
            }
        }
        wave_lds_fence();
      }
    });
    total += sum;
  }
  float acc[3], dv[3];
#pragma unroll
  for (int c = 0; c < 3; ++c) {
    acc[c] = __shfl(total, gr.base + c, 64);
    dv[c] = __shfl(total, gr.base + 3 + c, 64);
  }
  float disp = 0.f;
  if (valid && gr.rank == 0) disp = mom_epilogue<float, MODE>(a, i, local, acc, dv, D.vd);
  if (MODE != 0 && a.disp_out != nullptr) block_raise_max(a.disp_out, disp);
}

}  // namespace sph
