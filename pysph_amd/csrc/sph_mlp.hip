// Edge-MLP message-passing surrogate: forward, backward and Adam on the GPU.
//
// Network (per node i of a symmetric radius graph, hidden width 128):
//   H0   = ReLU(X_i W_in + b_in)                       X_i: 16 node features
//   for r in 1..2:
//     [P | Q] = H W_ab                                  (MFMA GEMM, N x 256)
//     A_i  = sum_j ReLU(P_i + Q_j + e_ij W_c + b_e)     e_ij: 16 edge features
//     U    = ReLU([H | A] W_u + c_u)                    (MFMA GEMM, N x 128)
//     H    = H + U
//   Y_i  = H_i W_out + b_out + a_i / g                  (2 outputs: acceleration / g)
// where a_i is the node's SPH pressure + artificial-viscosity acceleration
// (a parameter-free skip path kept in FP32): the network learns the
// correction that turns it into the acceleration over a 4x time step.
// Weights are kept in FP32 (Adam) with BF16 copies that feed the MFMA GEMMs
// (v_mfma_f32_32x32x16_bf16, FP32 accumulation).  Edge work is a fused
// gather / ReLU / sum per destination (one wave per node, its edges 32 at a
// time on the matrix cores); the backward pass recomputes the edge pre-activations and uses the
// graph's symmetry (j in N(i) <=> i in N(j)) to turn the scatter into Q's
// gradient into a gather.  Weight gradients are reduced through per-block
// partials, so every result is deterministic.
#include <algorithm>
#include <type_traits>
#include <vector>

#include "sph_internal.h"

namespace sph {
namespace mlp {

constexpr int kH = SPH_MLP_HIDDEN;   // 128
constexpr int kIn = SPH_MLP_NIN;     // 16 node features
constexpr int kE = SPH_MLP_NE;       // 16 edge features
constexpr int kR = SPH_MLP_ROUNDS;   // 2
constexpr int kOut = 2;

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

// ---- parameter layout (FP32 master; the BF16 copy uses the same offsets) --
struct Layout {
  int64_t w_in, b_in, w_ab[kR], w_c[kR], b_e[kR], w_u[kR], c_u[kR], w_out, b_out, total;
};
static Layout layout() {
  Layout L;
  int64_t o = 0;
  L.w_in = o; o += kIn * kH;
  L.b_in = o; o += kH;
  for (int r = 0; r < kR; ++r) {
    L.w_ab[r] = o; o += kH * 2 * kH;
    L.w_c[r] = o; o += kE * kH;
    L.b_e[r] = o; o += kH;
    L.w_u[r] = o; o += 2 * kH * kH;
    L.c_u[r] = o; o += kH;
  }
  L.w_out = o; o += kH * kOut;
  L.b_out = o; o += 4;
  L.total = o;
  return L;
}

// ---------------------------------------------------------------------------
// GEMM: C[M x N] = A[M x K] B[K x N] with B stored transposed ([N x K]), BF16
// operands, FP32 accumulate.  Block tile 64 x 64 (four 32 x 32 wave tiles).
// ---------------------------------------------------------------------------
struct GemmArgs {
  int M, N, K;
  const __bf16* A;
  int64_t lda;
  const __bf16* B;
  int64_t ldb;
  float* C;            // FP32 output (may be null)
  int64_t ldc;
  int accumulate;      // C += result
  float* C2;           // K = 128: when set, columns from n2 on are written here instead
  int64_t ldc2;        // of C (never accumulated)
  int n2;              // a multiple of 64: no block tile straddles it
  const float* bias;   // [N] or null
  int relu;
  float* U;            // activation before the residual (null: not stored)
  int64_t ldu;
  const float* res;    // residual added after the activation (null: none)
  int64_t ldr;
  __bf16* Cb;          // BF16 copy of the output (null: none)
  int64_t ldcb;
};

// Epilogue of the A B^T product with its loads issued ahead: the bias value
// of the lane's column once, and the residual and accumulated values of all
// 16 output elements before the first store, so that their latencies overlap
// (per element, each load would be waited for in turn).  Rows and columns
// past the matrix read row / column 0 and are not stored.  (v + bias, ReLU,
// U, + residual, + accumulated value, C, BF16 copy, in that order.)
struct EpiIn {
  int rows[16];  // output row of element r, -1 when outside the matrix
  float bv, rv[16], cv[16];
};

template <bool SPLIT = false>
__device__ __forceinline__ void epi_load(const GemmArgs& g, int orow0, int col, int lane,
                                         EpiIn& in) {
  const bool cok = col < g.N;
  const int ccol = cok ? col : 0;
  const bool acc = g.accumulate && !(SPLIT && col >= g.n2);
  in.bv = 0.f;
  if (g.bias) in.bv = g.bias[ccol];
#pragma unroll
  for (int r = 0; r < 16; ++r) {
    const int orow = orow0 + 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3);
    in.rows[r] = (cok && orow < g.M) ? orow : -1;
  }
  if (g.res) {
#pragma unroll
    for (int r = 0; r < 16; ++r)
      in.rv[r] = g.res[(int64_t)(in.rows[r] < 0 ? 0 : in.rows[r]) * g.ldr + ccol];
  }
  if (g.C && acc) {
#pragma unroll
    for (int r = 0; r < 16; ++r)
      in.cv[r] = g.C[(int64_t)(in.rows[r] < 0 ? 0 : in.rows[r]) * g.ldc + ccol];
  }
}

// Each output's flags are tested once, and a tile inside the matrix stores
// without a branch per element (43k rows: K = 128, N = 256 18.2 -> 15.9 us,
// K = 256, N = 128 20.5 -> 18.3; what is left is the rate of the stores,
// 44 MB and 33 MB).
template <bool SPLIT = false>
__device__ __forceinline__ void epi_store(const GemmArgs& g, const f32x16& acc, int col,
                                          const EpiIn& in) {
  const bool second = SPLIT && col >= g.n2;  // uniform over the block
  float* C = second ? g.C2 - g.n2 : g.C;
  const int64_t ldc = second ? g.ldc2 : g.ldc;
  float v[16];
#pragma unroll
  for (int r = 0; r < 16; ++r) {
    v[r] = acc[r];
    if (g.bias) v[r] += in.bv;
  }
  if (g.relu) {
#pragma unroll
    for (int r = 0; r < 16; ++r) v[r] = fmaxf(v[r], 0.f);
  }
  bool whole = true;
#pragma unroll
  for (int r = 0; r < 16; ++r) whole = whole && in.rows[r] >= 0;
  whole = __all(whole);
  auto put = [&](auto* out, int64_t ld) {
    out += col;
    if (whole) {
#pragma unroll
      for (int r = 0; r < 16; ++r)
        out[(int64_t)in.rows[r] * ld] = (std::remove_pointer_t<decltype(out)>)v[r];
    } else {
#pragma unroll
      for (int r = 0; r < 16; ++r)
        if (in.rows[r] >= 0)
          out[(int64_t)in.rows[r] * ld] = (std::remove_pointer_t<decltype(out)>)v[r];
    }
  };
  if (g.U) put(g.U, g.ldu);
  if (g.res) {
#pragma unroll
    for (int r = 0; r < 16; ++r) v[r] += in.rv[r];
  }
  if (C) {
    if (g.accumulate && !second) {
#pragma unroll
      for (int r = 0; r < 16; ++r) v[r] += in.cv[r];
    }
    put(C, ldc);
  }
  if (g.Cb) put(g.Cb, g.ldcb);
}

// C = A B^T-stored for K = 16 (the encoder): A [M x 16] row-major, B given as
// B^T [N x 16] row-major, so every fragment is one 16-byte load from global
// memory / L2.  Rows (columns) past M (N) load row (column) 0 and their
// outputs are not stored, so no load is predicated.
__global__ __launch_bounds__(256) void gemm_nt16_kernel(GemmArgs g) {
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int wm = w & 1, wn = w >> 1;
  const int row = blockIdx.y * 64 + wm * 32 + (lane & 31);
  const int col = blockIdx.x * 64 + wn * 32 + (lane & 31);
  const int kh = 8 * (lane >> 5);
  const bf16x8 a = *(const bf16x8*)(g.A + (int64_t)(row < g.M ? row : 0) * g.lda + kh);
  const bf16x8 b = *(const bf16x8*)(g.B + (int64_t)(col < g.N ? col : 0) * g.ldb + kh);
  f32x16 acc = {};
  acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, acc, 0, 0, 0);
  EpiIn in;
  epi_load(g, blockIdx.y * 64 + wm * 32, col, lane, in);
  epi_store(g, acc, col, in);
}

// The same product for K = 128 and 256 (forward layers with transposed BF16
// copies of the weights; input gradients with the weights themselves), both
// 64 x K tiles staged in LDS: the block loads A's
// 64 rows and B^T's 64 rows with 16-byte loads in which consecutive threads
// read consecutive bytes of a row (whole cache lines), then each wave reads
// its MFMA fragments from LDS.  Per-lane fragment loads from global memory
// touch 32 cache lines per instruction and kept the texture units 73 %
// busy.  The row pitch is K + 8 elements, so the eight 16-byte reads of a
// pass start 16 bytes apart modulo 128 (no bank conflicts).  Rows (columns)
// past M (N) load row (column) 0 and are not stored.  K = 16 KS (128 or 256:
// 35 or 68 KB of LDS).  SPLIT: columns from n2 on go to C2.
template <int KS, bool SPLIT = false>
__global__ __launch_bounds__(256) void gemm_nt_lds_kernel(GemmArgs g) {
  constexpr int K = 16 * KS;
  constexpr int kPitch = K + 8;
  constexpr int kPerRow = K / 8;  // 16-byte chunks per row
  __shared__ __align__(16) __bf16 sA[64 * kPitch];
  __shared__ __align__(16) __bf16 sB[64 * kPitch];
  const int tid = threadIdx.x;
  const int row0 = blockIdx.y * 64, col0 = blockIdx.x * 64;
#pragma unroll
  for (int i = 0; i < 64 * kPerRow / 256; ++i) {
    const int c = tid + 256 * i;
    const int r = c / kPerRow, kc = c % kPerRow;
    const int ar = row0 + r < g.M ? row0 + r : 0;
    const int bc = col0 + r < g.N ? col0 + r : 0;
    const bf16x8 va = *(const bf16x8*)(g.A + (int64_t)ar * g.lda + kc * 8);
    const bf16x8 vb = *(const bf16x8*)(g.B + (int64_t)bc * g.ldb + kc * 8);
    *(bf16x8*)(sA + r * kPitch + kc * 8) = va;
    *(bf16x8*)(sB + r * kPitch + kc * 8) = vb;
  }
  __syncthreads();
  const int lane = tid & 63, w = tid >> 6;
  const int wm = w & 1, wn = w >> 1;
  const int kh = 8 * (lane >> 5);
  const __bf16* ap = sA + (wm * 32 + (lane & 31)) * kPitch + kh;
  const __bf16* bp = sB + (wn * 32 + (lane & 31)) * kPitch + kh;
  f32x16 acc = {};
#pragma unroll
  for (int s = 0; s < KS; ++s) {
    const bf16x8 a = *(const bf16x8*)(ap + 16 * s);
    const bf16x8 b = *(const bf16x8*)(bp + 16 * s);
    acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, acc, 0, 0, 0);
  }
  const int col = col0 + wn * 32 + (lane & 31);
  EpiIn in;
  epi_load<SPLIT>(g, row0 + wm * 32, col, lane, in);
  epi_store<SPLIT>(g, acc, col, in);
}

// wt[n*K + k] = bf16(w[k*N + n]) for one K x N weight matrix.
__global__ __launch_bounds__(256) void transpose_bf16_kernel(int K, int N,
                                                             const float* __restrict__ w,
                                                             __bf16* __restrict__ wt) {
  const int t = blockIdx.x * 256 + threadIdx.x;
  if (t >= K * N) return;
  const int k = t / N, n = t % N;
  wt[(int64_t)n * K + k] = (__bf16)w[t];
}

// out[c] (+)= sum over z of part[z * zstride + c], c < cols: the fixed-order
// sum of per-block partials.  ZL lanes share a column: lane k sums slabs k,
// k + ZL, ... and the ZL partials are added as a tree in LDS.  One thread per
// column walking every slab was one chain of dependent memory waits: 179 us
// per launch on average over a training step of 33k nodes (up to 4096 slabs
// of 2176 columns); with the slabs shared out the same sums take 4-6 us.
template <int ZL>
__global__ __launch_bounds__(1024) void slab_sum_kernel(const float* __restrict__ part, int nslab,
                                                        int64_t zstride, int cols,
                                                        float* __restrict__ out, int acc) {
  constexpr int kCols = 1024 / ZL;
  __shared__ float red[ZL][kCols];
  const int t = threadIdx.x % kCols, k = threadIdx.x / kCols;
  const int c = blockIdx.x * kCols + t;
  float s = 0.f;
  if (c < cols) {
#pragma unroll 8
    for (int z = k; z < nslab; z += ZL) s += part[z * zstride + c];
  }
  red[k][t] = s;
  __syncthreads();
#pragma unroll
  for (int h = ZL / 2; h > 0; h >>= 1) {
    if (k < h) red[k][t] += red[k + h][t];
    __syncthreads();
  }
  if (k == 0 && c < cols) out[c] = acc ? out[c] + red[0][t] : red[0][t];
}

// Few slabs of many columns: one lane per column keeps every lane busy; many
// slabs: 16 columns a block, so that 64 lanes read each column's slabs (and
// a 64-byte segment of a slab at a time).
static void slab_sum(hipStream_t st, const float* part, int nslab, int64_t zstride, int cols,
                     float* out, int acc) {
  const dim3 b(1024);
  if (nslab <= 4)
    hipLaunchKernelGGL(slab_sum_kernel<1>, dim3((cols + 1023) / 1024), b, 0, st, part, nslab,
                       zstride, cols, out, acc);
  else if (nslab <= 128)
    hipLaunchKernelGGL(slab_sum_kernel<8>, dim3((cols + 127) / 128), b, 0, st, part, nslab,
                       zstride, cols, out, acc);
  else
    hipLaunchKernelGGL(slab_sum_kernel<64>, dim3((cols + 15) / 16), b, 0, st, part, nslab,
                       zstride, cols, out, acc);
}

// ---------------------------------------------------------------------------
// weight gradients: G[kdim x ncols] = X^T D over the rows (nodes)
// ---------------------------------------------------------------------------
struct GradArgs {
  int rows, kdim, ncols, chunk;  // chunk: rows per blockIdx.z, a multiple of 32
  const __bf16* X;               // [rows x kdim], leading dimension ldx
  int64_t ldx;
  const __bf16* D;               // [rows x ncols]
  int64_t ldd;
  float* part;                   // slab z at part + z * kdim * ncols
};

// Two rows of eight BF16 columns interleaved: out[c] = (row0[c], row1[c]).
__device__ __forceinline__ void interleave(const uint4 a, const uint4 b, uint32_t (&o)[8]) {
  const uint32_t av[4] = {a.x, a.y, a.z, a.w}, bv[4] = {b.x, b.y, b.z, b.w};
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    o[2 * i] = __builtin_amdgcn_perm(bv[i], av[i], 0x05040100);
    o[2 * i + 1] = __builtin_amdgcn_perm(bv[i], av[i], 0x07060302);
  }
}

// The contraction runs over the rows, so both operands would be read down
// their columns (the previous kernel: sixteen 2-byte loads per lane and
// MFMA, 118 us per product of 33k rows).  Here a block owns a TM x TN tile
// of G and a chunk of rows; it loads 32 rows at a time in whole 16-byte
// pieces, interleaves pairs of rows in registers, and keeps the pair (rows
// 2p, 2p + 1) of column c as one dword at lds[p][c]: an MFMA fragment of a
// column (rows 8h..8h+7 of a 16-row step for half-wave h) is then four
// conflict-free 4-byte LDS reads.  The next 32 rows are loaded into
// registers while the current ones are multiplied.  Rows past the chunk are
// zeros, columns past the matrix are loaded from column 0 and not stored.
// TM x TN is 128 x 64 (32 x 128 for the 16 node features).
template <int TM, int TN>
__global__ __launch_bounds__(256) void grad_kernel(GradArgs g) {
  constexpr int kRows = 32, kPairs = kRows / 2;
  constexpr int kCx = TM / 8, kCd = TN / 8;   // 16-byte pieces per row
  constexpr int WM = TM >= 128 ? 2 : 1, WN = 4 / WM;  // wave grid
  constexpr int FM = TM / (32 * WM), FN = TN / (32 * WN);
  constexpr int kTasks = kPairs * (kCx + kCd);
  constexpr int kPer = (kTasks + 255) / 256;
  static_assert(FM >= 1 && FN >= 1 && FM * 32 * WM == TM && FN * 32 * WN == TN, "tile");
  // 16 dwords of padding: the pitch stays a multiple of four dwords for the
  // 16-byte writes and consecutive pairs start 16 banks apart
  __shared__ __align__(16) uint32_t lds[kPairs][TM + TN + 16];
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  const int m0 = blockIdx.y * TM, n0 = blockIdx.x * TN;
  const int r_begin = blockIdx.z * g.chunk, r_end = min(g.rows, r_begin + g.chunk);
  uint4 va[kPer], vb[kPer];
  auto load = [&](int r0) {
#pragma unroll
    for (int i = 0; i < kPer; ++i) {
      const int t = tid + 256 * i;
      va[i] = vb[i] = make_uint4(0, 0, 0, 0);
      if (t >= kTasks) continue;
      const int p = t / (kCx + kCd), c = t % (kCx + kCd);
      const bool x = c < kCx;
      const int col = x ? m0 + 8 * c : n0 + 8 * (c - kCx);
      const __bf16* base = x ? g.X : g.D;
      const int64_t ld = x ? g.ldx : g.ldd;
      const int cc = col < (x ? g.kdim : g.ncols) ? col : 0;
      const int r = r0 + 2 * p;
      if (r < r_end) va[i] = *(const uint4*)(base + (int64_t)r * ld + cc);
      if (r + 1 < r_end) vb[i] = *(const uint4*)(base + (int64_t)(r + 1) * ld + cc);
    }
  };
  f32x16 acc[FM][FN] = {};
  load(r_begin);
  for (int r0 = r_begin; r0 < r_end; r0 += kRows) {
    __syncthreads();
#pragma unroll
    for (int i = 0; i < kPer; ++i) {
      const int t = tid + 256 * i;
      if (t >= kTasks) continue;
      const int p = t / (kCx + kCd), c = t % (kCx + kCd);
      uint32_t o[8];
      interleave(va[i], vb[i], o);
      *(uint4*)&lds[p][8 * c] = make_uint4(o[0], o[1], o[2], o[3]);
      *(uint4*)&lds[p][8 * c + 4] = make_uint4(o[4], o[5], o[6], o[7]);
    }
    __syncthreads();
    if (r0 + kRows < r_end) load(r0 + kRows);
    const int wm = w % WM, wn = w / WM;
#pragma unroll
    for (int s = 0; s < kRows / 16; ++s) {
      const int p0 = 8 * s + 4 * (lane >> 5);
      bf16x8 a[FM], b[FN];
      auto frag = [&](int col) {
        union {
          uint32_t u[4];
          bf16x8 v;
        } f;
#pragma unroll
        for (int k = 0; k < 4; ++k) f.u[k] = lds[p0 + k][col];
        return f.v;
      };
#pragma unroll
      for (int i = 0; i < FM; ++i) a[i] = frag((wm * FM + i) * 32 + (lane & 31));
#pragma unroll
      for (int j = 0; j < FN; ++j) b[j] = frag(TM + (wn * FN + j) * 32 + (lane & 31));
#pragma unroll
      for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j)
          acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[i], b[j], acc[i][j], 0, 0, 0);
    }
  }
  float* out = g.part + (int64_t)blockIdx.z * g.kdim * g.ncols;
  const int wm = w % WM, wn = w / WM;
#pragma unroll
  for (int i = 0; i < FM; ++i)
#pragma unroll
    for (int j = 0; j < FN; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int row = m0 + (wm * FM + i) * 32 + 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3);
        const int col = n0 + (wn * FN + j) * 32 + (lane & 31);
        if (row < g.kdim && col < g.ncols) out[(int64_t)row * g.ncols + col] = acc[i][j][r];
      }
}

// ---------------------------------------------------------------------------
// features
// ---------------------------------------------------------------------------
struct FeatArgs {
  int n;
  const float4* pos4;
  const float4* vel4;
  const float* rho;
  const int* btype;
  const int64_t* off;
  const int64_t* nbr;
  int64_t ne;  // entries of nbr, see edge_end
  float rho0, co, gamma, B, u_scale, g, rho_scale, alpha, eta;
  int dim;
};

// CSR offset `o` of a graph with room for `ne` edges.  A build that found
// more (sph_neighbor_fill_capped flags it, the caller reads the flag later)
// leaves offsets past the room: rows end there, so that no kernel reads
// neighbours or features that were never written.
__device__ __forceinline__ int64_t edge_end(int64_t o, int64_t ne) { return o < ne ? o : ne; }

__device__ __forceinline__ float tait_p(const FeatArgs& f, float rho) {
  return f.B * (powf(rho / f.rho0, f.gamma) - 1.f);
}

// Cubic spline W and grad factor of the 2D/3D kernel (kernels.pyx:367-412),
// h = the pair's mean smoothing length.
__device__ __forceinline__ void spline(float r, float h, int dim, float& w, float& gf) {
  const float q = r / h;
  const float fac = dim == 2 ? 10.f / (7.f * 3.14159265358979f * h * h)
                             : 1.f / (3.14159265358979f * h * h * h);
  const float t = 2.f - q;
  if (q > 2.f) {
    w = 0.f;
    gf = 0.f;
  } else if (q > 1.f) {
    w = fac * 0.25f * t * t * t;
    gf = fac * (-0.75f * t * t / (h * r));
  } else {
    w = fac * (1.f - 1.5f * q * q * (1.f - 0.5f * q));
    gf = q > 1e-14f ? fac * 3.f * (0.75f * q - 1.f) / (h * h) : 0.f;
  }
}

// Node features: u/U, v/U, (rho/rho0 - 1) S, p/B, boundary flag, 1, and the
// node's SPH pressure and artificial-viscosity accelerations / g (the sums
// over its edges, from edge_feat_kernel).
__global__ __launch_bounds__(256) void node_feat_kernel(FeatArgs f, const float* __restrict__ acc4,
                                                        __bf16* __restrict__ X) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i >= f.n) return;
  const float4 v = f.vel4[i];
  const float rho = f.rho[i];
  float x[kIn] = {};
  x[0] = v.x / f.u_scale;
  x[1] = v.y / f.u_scale;
  x[2] = (rho / f.rho0 - 1.f) * f.rho_scale;
  x[3] = tait_p(f, rho) / f.B;
  x[4] = f.btype[i] ? 1.f : 0.f;
  x[5] = 1.f;
  // the SPH accelerations enter the network scaled down (they reach 100s of
  // g at a summation-density free surface); the decoder's skip path adds
  // them unscaled
#pragma unroll
  for (int c = 0; c < 4; ++c) x[6 + c] = 0.01f * acc4[(int64_t)i * 4 + c];
#pragma unroll
  for (int k = 0; k < kIn; ++k) X[(int64_t)i * kIn + k] = (__bf16)x[k];
}

// Edge features of edge (i <- j), one lane per edge.  Antisymmetric parts
// change sign and the rho_i / rho_j slots swap for the reverse edge
// (see reverse_feat), which the backward pass relies on.
// kFeatLanes lanes per node: a node has about 21 edges in 2D, so a whole
// wave per node would leave two thirds of its lanes idle (the features
// launch 0.077 -> 0.048 ms on the 64k-particle dam break)
constexpr int kFeatLanes = 16;
constexpr int kFeatNodes = 256 / kFeatLanes;  // nodes per 256-thread block

__global__ __launch_bounds__(256) void edge_feat_kernel(FeatArgs f, float* __restrict__ E,
                                                        float* __restrict__ acc4) {
  const int i = blockIdx.x * kFeatNodes + (int)(threadIdx.x / kFeatLanes);
  const int lane = threadIdx.x % kFeatLanes;
  // every lane stays for the group reductions below (no early return)
  const bool node = i < f.n;
  const int64_t e0 = node ? edge_end(f.off[i], f.ne) : 0;
  const int64_t e1 = node ? edge_end(f.off[i + 1], f.ne) : 0;
  const float4 pi = f.pos4[node ? i : 0], vi = f.vel4[node ? i : 0];
  const float ri = f.rho[node ? i : 0];
  const float pri = tait_p(f, ri);
  float sum[4] = {0.f, 0.f, 0.f, 0.f};
  for (int64_t e = e0 + lane; e < e1; e += kFeatLanes) {
    const int j = (int)f.nbr[e];
    const float4 pj = f.pos4[j], vj = f.vel4[j];
    const float rj = f.rho[j];
    const float prj = tait_p(f, rj);
    const float h = 0.5f * (pi.w + pj.w);
    const float dx = pi.x - pj.x, dy = pi.y - pj.y, dz = pi.z - pj.z;
    const float r = sqrtf(dx * dx + dy * dy + dz * dz);
    float w, gf;
    spline(r, h, f.dim, w, gf);
    const float du = vi.x - vj.x, dv = vi.y - vj.y, dw = vi.z - vj.z;
    const float mbar = 0.5f * (vi.w + vj.w);
    const float pt = -mbar * (pri / (ri * ri) + prj / (rj * rj)) * gf / f.g;
    const float dot = du * dx + dv * dy + dw * dz;
    float visc = 0.f;
    if (dot < 0.f) {
      const float cbar = 0.5f * f.co * (powf(ri / f.rho0, 0.5f * (f.gamma - 1.f)) +
                                        powf(rj / f.rho0, 0.5f * (f.gamma - 1.f)));
      const float mu = h * dot / (r * r + f.eta * f.eta * h * h);
      visc = -mbar * (-f.alpha * cbar * mu) / (0.5f * (ri + rj)) * gf / f.g;
    }
    sum[0] += pt * dx;
    sum[1] += pt * dy;
    sum[2] += visc * dx;
    sum[3] += visc * dy;
    // a pair's pressure term is of order (p/rho)/h ~ g H / h; scale to O(1)
    const float ps = 2.f * f.g * h / (f.u_scale * f.u_scale);
    float x[kE] = {};
    x[0] = dx / h;
    x[1] = dy / h;
    x[2] = r / h;
    x[3] = du / f.u_scale;
    x[4] = dv / f.u_scale;
    x[5] = (ri / f.rho0 - 1.f) * f.rho_scale;
    x[6] = (rj / f.rho0 - 1.f) * f.rho_scale;
    x[7] = w * h * h;
    x[8] = pt * dx * ps;
    x[9] = pt * dy * ps;
    x[10] = visc * dx * ps;
    x[11] = visc * dy * ps;
    x[12] = 1.f;
#pragma unroll
    for (int k = 0; k < kE; ++k) E[e * kE + k] = x[k];
  }
#pragma unroll
  for (int c = 0; c < 4; ++c) {
    float v = sum[c];
    for (int off = kFeatLanes / 2; off > 0; off >>= 1) v += __shfl_xor(v, off, kFeatLanes);
    if (lane == 0 && node) acc4[(int64_t)i * 4 + c] = v;
  }
}

// Features of edge (j <- i) from those of (i <- j).
__device__ __forceinline__ float reverse_feat(const float* x, int k) {
  switch (k) {
    case 0: case 1: case 3: case 4: case 8: case 9: case 10: case 11: return -x[k];
    case 5: return x[6];
    case 6: return x[5];
    default: return x[k];
  }
}

// ---------------------------------------------------------------------------
// message passing (one wave per destination node, channels lane, lane + 64)
// ---------------------------------------------------------------------------
struct EdgeArgs {
  int n;
  const int64_t* off;
  const int64_t* nbr;
  int64_t ne;           // entries of nbr and rows of E, see edge_end
  const float* E;       // [edges x kE]
  const float* PQ;      // [n x 2H]: P | Q
  const float* Wc;      // [kE x H]
  const float* be;      // [H]
  __bf16* A;            // forward: aggregate written at A + i*lda (BF16)
  int64_t lda;
  // backward
  const float* dA;      // [n x ldda] gradient of the aggregate
  int64_t ldda;
  __bf16* dPQb;         // [n x 2H]: dP | dQ, rounded to BF16
  float* part;          // [slabs x (kE + 1) x H] partial dWc, dbe
};

__global__ __launch_bounds__(256) void edge_fwd_kernel(EdgeArgs a) {
  const int i = __builtin_amdgcn_readfirstlane(blockIdx.x * 4 + (threadIdx.x >> 6));
  const int lane = threadIdx.x & 63;
  if (i >= a.n) return;
  float wc0[kE], wc1[kE];
#pragma unroll
  for (int k = 0; k < kE; ++k) {
    wc0[k] = a.Wc[k * kH + lane];
    wc1[k] = a.Wc[k * kH + lane + 64];
  }
  const float p0 = a.PQ[(int64_t)i * 2 * kH + lane] + a.be[lane];
  const float p1 = a.PQ[(int64_t)i * 2 * kH + lane + 64] + a.be[lane + 64];
  float s0 = 0.f, s1 = 0.f;
  const int64_t e0 = edge_end(a.off[i], a.ne), e1 = edge_end(a.off[i + 1], a.ne);
  // four edges per iteration: their neighbour rows are in flight together
  constexpr int U = 4;
  for (int64_t e = e0; e < e1; e += U) {
    float q0[U], q1[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int64_t eu = e + u < e1 ? e + u : e0;
      const int j = (int)a.nbr[eu];
      q0[u] = a.PQ[(int64_t)j * 2 * kH + kH + lane];
      q1[u] = a.PQ[(int64_t)j * 2 * kH + kH + lane + 64];
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      if (e + u >= e1) break;
      const float* x = a.E + (e + u) * kE;
      float z0 = p0 + q0[u], z1 = p1 + q1[u];
#pragma unroll
      for (int k = 0; k < kE; ++k) {
        const float xk = x[k];
        z0 += xk * wc0[k];
        z1 += xk * wc1[k];
      }
      s0 += fmaxf(z0, 0.f);
      s1 += fmaxf(z1, 0.f);
    }
  }
  a.A[(int64_t)i * a.lda + lane] = (__bf16)s0;
  a.A[(int64_t)i * a.lda + lane + 64] = (__bf16)s1;
}

#ifndef SPH_EDGE_MFMA
#define SPH_EDGE_MFMA 1
#endif

// x = hi + lo with hi = bf16(x) and lo = bf16(x - hi): hi*w_hi + hi*w_lo +
// lo*w_hi reproduces an FP32 product to ~2^-16 relative.
__device__ __forceinline__ void split_bf16(float x, __bf16& hi, __bf16& lo) {
  hi = (__bf16)x;
  lo = (__bf16)(x - (float)hi);
}

// The aggregation A_i = sum_j ReLU(P_i + b + Q_j + e_ij W_c) on the matrix
// cores.  A wave takes the edges of node i 32 at a time: the 32 x 16 block
// of edge features times W_c (16 x 128) is four v_mfma_f32_32x32x16_bf16
// tiles of 32 hidden units, each as three products of the features' and
// W_c's BF16 high and low parts (the FP32 products to ~2^-16).  In the
// product's layout, lane l holds hidden unit 32t + (l & 31) of the 16 edge
// rows 8(r / 4) + 4(l / 32) + (r % 4); it adds P_i + b, then Q_j, applies the
// ReLU and sums its rows one after another, and the two half-waves' row sums
// are added at the end.  That order is part of the result: A is stored in
// BF16, where a last bit of a sum can become 2^-8 of a value, and a
// surrogate run carries it through all of its steps.  The block splits W_c
// into its BF16 fragments in LDS once (8 KB, in the lanes' fragment order, so
// each read is one conflict-free ds_read_b128); then its waves take the nodes
// of the block's run (node_run) in turn.
//
// Bound by the return of neighbour rows from L1 (21 edges of 512 B a node in
// 2D: TD 73 % busy) beside its vector instructions, so the matrix cores take
// the masks: rows past the node's last edge (which re-read that edge) get
// kPastEnd through feature slot 13, one of the three that edge_feat_kernel
// leaves zero, and so leave the ReLU as 0.  Neighbour rows are addressed by
// 32-bit byte offsets from the uniform base.  The rows of the next tile are in
// flight while a tile is summed, the next block's features and indices while
// the last two tiles are.  43k nodes, 0.9M edges: 59 us with a mask per
// element and nothing loaded ahead, 45.4 so (46.7 with three waves per SIMD,
// five spill; with Q_j as the products' initial accumulator and two
// interleaved sums, which round differently, 44.5).
#ifndef SPH_EDGE_WAVES
#define SPH_EDGE_WAVES 4
#endif
constexpr float kPastEnd = -8.507059173e37f;  // -2^126, a BF16 value
constexpr int kPastSlot = 13;

// The nodes of one block of a persistent edge kernel: a run of consecutive
// (cell-ordered) nodes, whose neighbourhoods overlap, taken in turn by the
// block's four waves; an XCD's blocks get neighbouring runs.
struct NodeRun {
  int lo, hi;
};
__device__ __forceinline__ NodeRun node_run(int n) {
  const int nb = gridDim.x, lb = xcd_block(blockIdx.x, nb);
  const int per = n / nb, rem = n % nb;  // block lb has per + (lb < rem) nodes
  const int lo = lb * per + (lb < rem ? lb : rem);
  return {lo, lo + per + (lb < rem ? 1 : 0)};
}

// v is complete here and no later load starts before: without it the sums
// of all tiles move behind all of their loads.
__device__ __forceinline__ void hold_order(float& v) {
  asm volatile("" : "+v"(v)::"memory");
  __builtin_amdgcn_sched_barrier(0);
}

// The next 32 edges of a wave: the lane's half of edge row m's features and
// the row's neighbour.  A node without edges reads some edge of the graph,
// which has at least one, and sums none.
struct EdgeRows {
  float4 x0, x1;
  int j;
};
__device__ __forceinline__ EdgeRows edge_rows(const EdgeArgs& a, int64_t e0, int64_t e1, int m,
                                              int kh) {
  EdgeRows x;
  const int64_t e = e0 + m < e1 ? e0 + m : (e1 > 0 ? e1 - 1 : 0);
  x.x0 = *(const float4*)(a.E + e * kE + kh);
  x.x1 = *(const float4*)(a.E + e * kE + kh + 4);
  x.j = (int)a.nbr[e];
  return x;
}

// One block of up to 32 edges: the four tiles' products and sums, with the
// next block's features, neighbours and P row loaded on the way.  (Leaving
// out the eights of rows past the last edge, in copies of this for 16 and 24
// edges, gained nothing.)
__device__ __forceinline__ EdgeRows edge_block(const EdgeArgs& a, int64_t ne0, int64_t ne1, int pi,
                                               int m, int kh, const unsigned (&qoff)[16],
                                               bf16x8 ah, bf16x8 al, const bf16x8* wfrag,
                                               const float (&pb)[4], float (&sum)[4],
                                               float (&pn)[4]) {
  const char* const Qb = (const char*)(a.PQ + kH);
  const int lane = threadIdx.x & 63;
  EdgeRows x;
  float q[2][16];
#pragma unroll
  for (int r = 0; r < 16; ++r) q[0][r] = *(const float*)(Qb + qoff[r]);
  hold_order(sum[0]);  // not mixed with the next tile's
#pragma unroll
  for (int t = 0; t < 4; ++t) {
    if (t < 3) {
#pragma unroll
      for (int r = 0; r < 16; ++r)
        q[(t + 1) & 1][r] = *(const float*)(Qb + 128 * (t + 1) + qoff[r]);
    }
    if (t == 2) {
#pragma unroll
      for (int c = 0; c < 4; ++c) pn[c] = a.PQ[(int64_t)pi * 2 * kH + 32 * c + m];
      x = edge_rows(a, ne0, ne1, m, kh);
    }
    // one tile's rows in flight ahead, not all of them
    __builtin_amdgcn_sched_barrier(0);
    const bf16x8 bh = wfrag[t * 64 + lane], bl = wfrag[256 + t * 64 + lane];
    f32x16 z = {};
    z = __builtin_amdgcn_mfma_f32_32x32x16_bf16(al, bh, z, 0, 0, 0);
    z = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ah, bl, z, 0, 0, 0);
    z = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ah, bh, z, 0, 0, 0);
#pragma unroll
    for (int r = 0; r < 16; ++r) sum[t] += fmaxf((z[r] + pb[t]) + q[t & 1][r], 0.f);
    hold_order(sum[t]);
  }
  return x;
}

__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(SPH_EDGE_WAVES)))
void edge_fwd_mfma_kernel(EdgeArgs a, const int64_t* __restrict__ off) {
  const int n = a.n;
  const float* const PQ = a.PQ;
  __bf16* const A = a.A;
  const int64_t lda = a.lda;
  __shared__ bf16x8 wfrag[2 * 4 * 64];  // [hi, lo][tile][lane]
  for (int f = threadIdx.x; f < 2 * 4 * 64; f += 256) {
    const int l = f & 63, t = (f >> 6) & 3, lo = f >> 8;
    const int c = 32 * t + (l & 31), k0 = 8 * (l >> 5);
    bf16x8 v;
#pragma unroll
    for (int s = 0; s < 8; ++s) {
      __bf16 h, l2;
      split_bf16(a.Wc[(k0 + s) * kH + c], h, l2);
      v[s] = lo ? l2 : h;
      if (k0 + s >= kPastSlot)
        v[s] = (__bf16)(k0 + s == kPastSlot && !lo ? kPastEnd : 0.f);
    }
    wfrag[f] = v;
  }
  __syncthreads();
  const int lane = threadIdx.x & 63;
  const NodeRun run = node_run(n);
  int i = __builtin_amdgcn_readfirstlane(run.lo + (int)(threadIdx.x >> 6));
  if (i >= run.hi) return;
  if (edge_end(off[n], a.ne) <= 0) {  // a graph without edges
    for (; i < run.hi; i += 4) {
      A[(int64_t)i * lda + lane] = (__bf16)0.f;
      A[(int64_t)i * lda + 64 + lane] = (__bf16)0.f;
    }
    return;
  }
  const int m = lane & 31, kh = 8 * (lane >> 5);
  const int mr0 = 4 * (lane >> 5);  // edge row of r is mr0 + 8(r / 4) + r % 4
  float be[4], pn[4], pb[4], sum[4] = {};
#pragma unroll
  for (int t = 0; t < 4; ++t) {
    be[t] = a.be[32 * t + m];
    pn[t] = PQ[(int64_t)i * 2 * kH + 32 * t + m];
  }
  int64_t e0 = edge_end(off[i], a.ne), e1 = edge_end(off[i + 1], a.ne);
  EdgeRows x = edge_rows(a, e0, e1, m, kh);
  bool first = true;  // first block of node i
  // as many stores behind the loads as at the loop's end, so that its top
  // waits for the loads alone (the same lanes overwrite them)
  const int cl = lane + (kh ? 32 : 0);
  A[(int64_t)i * lda + cl] = (__bf16)0.f;
  A[(int64_t)i * lda + cl + 32] = (__bf16)0.f;
  for (;;) {
    // the block after this one (past the last node: this one again, unused)
    const bool last = e0 + 32 >= e1;
    const int ni = last ? i + 4 : i;
    const bool more = ni < run.hi;
    const int64_t ne0 = last ? edge_end(off[more ? ni : i], a.ne) : e0 + 32;
    const int64_t ne1 = last ? edge_end(off[(more ? ni : i) + 1], a.ne) : e1;
    const int lim = (int)(e1 - e0);  // rows below lim are edges of node i
    if (first) {
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        pb[t] = pn[t] + be[t];
        sum[t] = 0.f;
      }
    }
    unsigned qoff[16];  // byte offset of Q_j's element m, edge row r
#pragma unroll
    for (int r = 0; r < 16; ++r)
      qoff[r] = ((unsigned)__shfl(x.j, mr0 + 8 * (r >> 2) + (r & 3)) * 2 * kH + m) * 4;
    const float xs[8] = {x.x0.x, x.x0.y, x.x0.z, x.x0.w, x.x1.x, x.x1.y, x.x1.z, x.x1.w};
    bf16x8 ah, al;
#pragma unroll
    for (int s = 0; s < 8; ++s) {
      __bf16 h, l;
      split_bf16(xs[s], h, l);
      if (s == kPastSlot - 8 && kh) h = (__bf16)(m < lim ? 0.f : 1.f);
      ah[s] = h;
      al[s] = l;
    }
    x = edge_block(a, ne0, ne1, more ? ni : i, m, kh, qoff, ah, al, wfrag, pb, sum, pn);
    first = last;
    // stored after every block, whole after the node's last one: without a
    // branch around the stores, the loads above need not wait for them
    float tot[4];
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      tot[t] = sum[t] + __shfl_xor(sum[t], 32);
      if (lim <= 0) tot[t] = 0.f;  // no edges
    }
    __bf16* const Ai = A + (int64_t)i * lda + cl;
    Ai[0] = (__bf16)(kh ? tot[2] : tot[0]);
    Ai[32] = (__bf16)(kh ? tot[3] : tot[1]);
    if (!more) return;
    i = ni;
    e0 = ne0;
    e1 = ne1;
  }
}

// Persistent: each wave walks nodes i = wave, wave + nwaves, ...  and keeps
// its dWc / dbe partial sums in registers.
__global__ __launch_bounds__(256) void edge_bwd_kernel(EdgeArgs a) {
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(blockIdx.x * 4 + (threadIdx.x >> 6));
  const int nwaves = gridDim.x * 4;
  float wc0[kE], wc1[kE], g0[kE], g1[kE];
#pragma unroll
  for (int k = 0; k < kE; ++k) {
    wc0[k] = a.Wc[k * kH + lane];
    wc1[k] = a.Wc[k * kH + lane + 64];
    g0[k] = 0.f;
    g1[k] = 0.f;
  }
  const float be0 = a.be[lane], be1 = a.be[lane + 64];
  float gb0 = 0.f, gb1 = 0.f;
  for (int i = wave; i < a.n; i += nwaves) {
    const float* PQi = a.PQ + (int64_t)i * 2 * kH;
    const float pi0 = PQi[lane] + be0, pi1 = PQi[lane + 64] + be1;
    const float qi0 = PQi[kH + lane], qi1 = PQi[kH + lane + 64];
    const float dai0 = a.dA[(int64_t)i * a.ldda + lane];
    const float dai1 = a.dA[(int64_t)i * a.ldda + lane + 64];
    float dp0 = 0.f, dp1 = 0.f, dq0 = 0.f, dq1 = 0.f;
    const int64_t e0 = edge_end(a.off[i], a.ne), e1 = edge_end(a.off[i + 1], a.ne);
    for (int64_t e = e0; e < e1; ++e) {
      const int j = (int)a.nbr[e];
      const float* x = a.E + e * kE;
      const float* PQj = a.PQ + (int64_t)j * 2 * kH;
      // edge (i <- j): s = P_i + Q_j + e_ij Wc + b
      float s0 = pi0 + PQj[kH + lane], s1 = pi1 + PQj[kH + lane + 64];
      // edge (j <- i): s' = P_j + Q_i + e_ji Wc + b
      float t0 = PQj[lane] + be0 + qi0, t1 = PQj[lane + 64] + be1 + qi1;
      float xk[kE];
#pragma unroll
      for (int k = 0; k < kE; ++k) xk[k] = x[k];
#pragma unroll
      for (int k = 0; k < kE; ++k) {
        s0 += xk[k] * wc0[k];
        s1 += xk[k] * wc1[k];
        const float rk = reverse_feat(xk, k);
        t0 += rk * wc0[k];
        t1 += rk * wc1[k];
      }
      const float ds0 = s0 > 0.f ? dai0 : 0.f, ds1 = s1 > 0.f ? dai1 : 0.f;
      dp0 += ds0;
      dp1 += ds1;
#pragma unroll
      for (int k = 0; k < kE; ++k) {
        g0[k] += xk[k] * ds0;
        g1[k] += xk[k] * ds1;
      }
      gb0 += ds0;
      gb1 += ds1;
      const float daj0 = a.dA[(int64_t)j * a.ldda + lane];
      const float daj1 = a.dA[(int64_t)j * a.ldda + lane + 64];
      dq0 += t0 > 0.f ? daj0 : 0.f;
      dq1 += t1 > 0.f ? daj1 : 0.f;
    }
    __bf16* db = a.dPQb + (int64_t)i * 2 * kH;
    db[lane] = (__bf16)dp0;
    db[lane + 64] = (__bf16)dp1;
    db[kH + lane] = (__bf16)dq0;
    db[kH + lane + 64] = (__bf16)dq1;
  }
  float* p = a.part + (int64_t)wave * (kE + 1) * kH;
#pragma unroll
  for (int k = 0; k < kE; ++k) {
    p[k * kH + lane] = g0[k];
    p[k * kH + lane + 64] = g1[k];
  }
  p[kE * kH + lane] = gb0;
  p[kE * kH + lane + 64] = gb1;
}

// The same on the matrix cores.  A wave takes node i's edges 32 at a time, in
// the layout of the forward aggregation (lane l: hidden unit 32t + (l & 31) of
// 16 edge rows).  Per tile of 32 hidden units:
//   s = Q_j + e_ij Wc and t = P_j + e_ji Wc: products whose initial
//     accumulators are the gathered rows.  e_ji Wc is e_ij times Wc with its
//     rows' signs and places changed as reverse_feat changes the features'.
//     The signs of s + P_i + b and t + Q_i + b are compared without the sum.
//     They decide the masks, so the products are FP32 ones: three BF16 parts
//     hold a feature or a weight exactly, and six of their nine products
//     leave 2^-27 of one (the forward pass's two parts: 2^-16).  Rms error of
//     a pre-activation against 64 bits, on a million random edges with terms
//     of order 1: 7.5e-8; one FMA after another: 1.8e-7; two parts: 2.8e-6.
//   dQ_i: the lane's dA_j of the rows whose t is positive, summed.
//   dWc: dA_i is one value for all of the node's edges, so the sum over them
//     is dA_i * (x^T mask): a product with the 0 / 1 mask of s, which BF16
//     holds exactly, and x as three BF16 parts (the FP32 features, exactly):
//     rows 0-15 of the first product are the high parts, 16-31 the middle
//     ones, rows 0-15 of the second the low ones.  The mask needs no move
//     between lanes: the 8 rows a lane holds are a product's 8 depth slots when
//     x^T is read in the same row order.  Feature slot 13, always zero, is
//     one here: its row counts the masked edges (dP_i = count * dA_i, dbe).
// Rows past the last edge are pushed below zero as in the forward pass.
// dWc is kept in registers and summed over the block's waves at the end.
// Bound by the return of gathered rows from L1 (1.5 KB an edge: TD 83 % busy);
// vector arithmetic alone (110 FP32 instructions per edge and wave) took
// 156 us for 33k nodes, this 124 (112 with two parts in s and t).  Loading a tile's rows ahead gained
// nothing, leaving out rows past the last edge spilled.
__device__ __forceinline__ void split3_bf16(float x, __bf16& h, __bf16& m, __bf16& l) {
  h = (__bf16)x;
  const float d = x - (float)h;
  m = (__bf16)d;
  l = (__bf16)(d - (float)m);
}

// Row of Wc that feature k multiplies in the reverse edge, and its sign.
__device__ __forceinline__ int reverse_row(int k) { return k == 5 ? 6 : (k == 6 ? 5 : k); }
__device__ __forceinline__ float reverse_sign(int k) {
  return k == 0 || k == 1 || k == 3 || k == 4 || (k >= 8 && k <= 11) ? -1.f : 1.f;
}

// c + x w of the parts of x (ah, am, al) and w (wf: high, middle and low
// fragments 256 apart), smallest products first.
__device__ __forceinline__ f32x16 edge_product(bf16x8 ah, bf16x8 am, bf16x8 al, const bf16x8* wf,
                                               f32x16 c) {
  const bf16x8 wh = wf[0], wm = wf[256], wl = wf[512];
  c = __builtin_amdgcn_mfma_f32_32x32x16_bf16(al, wh, c, 0, 0, 0);
  c = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ah, wl, c, 0, 0, 0);
  c = __builtin_amdgcn_mfma_f32_32x32x16_bf16(am, wm, c, 0, 0, 0);
  c = __builtin_amdgcn_mfma_f32_32x32x16_bf16(am, wh, c, 0, 0, 0);
  c = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ah, wm, c, 0, 0, 0);
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(ah, wh, c, 0, 0, 0);
}

constexpr int kBwdWaves = 2;  // per SIMD
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(kBwdWaves)))
void edge_bwd_mfma_kernel(EdgeArgs a, const int64_t* __restrict__ off) {
  __shared__ bf16x8 wfrag[6 * 4 * 64];  // [s, t][high, middle, low part][tile][lane]
  __shared__ float slab[(kE + 1) * kH];
  for (int f = threadIdx.x; f < 6 * 4 * 64; f += 256) {
    const int l = f & 63, t = (f >> 6) & 3, part = (f >> 8) % 3, rev = (f >> 8) / 3;
    const int c = 32 * t + (l & 31), k0 = 8 * (l >> 5);
    bf16x8 v;
#pragma unroll
    for (int s = 0; s < 8; ++s) {
      const int k = k0 + s;
      const float w = rev ? reverse_sign(k) * a.Wc[reverse_row(k) * kH + c] : a.Wc[k * kH + c];
      __bf16 h, md, lo;
      split3_bf16(w, h, md, lo);
      v[s] = part == 0 ? h : (part == 1 ? md : lo);
      if (k >= kPastSlot) v[s] = (__bf16)(k == kPastSlot && part == 0 ? kPastEnd : 0.f);
    }
    wfrag[f] = v;
  }
  for (int f = threadIdx.x; f < (kE + 1) * kH; f += 256) slab[f] = 0.f;
  __syncthreads();
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const int m = lane & 31, hf = lane >> 5, kh = 8 * hf;
  const int mr0 = 4 * hf;  // edge row of r is mr0 + 8(r / 4) + r % 4
  const int fk = m & 15;   // feature of this lane's row of x^T
  const char* const Pb = (const char*)a.PQ;
  const char* const Db = (const char*)a.dA;
  const unsigned dpitch = (unsigned)a.ldda * 4;
  float be[4], gt[4][8];  // gt[t][r]: feature 8(r / 4) + mr0 + r % 4, hidden unit 32t + m
#pragma unroll
  for (int t = 0; t < 4; ++t) {
    be[t] = a.be[32 * t + m];
#pragma unroll
    for (int r = 0; r < 8; ++r) gt[t][r] = 0.f;
  }
  const NodeRun run = node_run(a.n);
  for (int i = __builtin_amdgcn_readfirstlane(run.lo + wv); i < run.hi; i += 4) {
    const int64_t e0 = edge_end(off[i], a.ne), e1 = edge_end(off[i + 1], a.ne);
    float npb[4], nqb[4], dai[4], dq[4], cnt[4];  // npb = -(P_i + b), nqb = -(Q_i + b)
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      const float* p = a.PQ + (int64_t)i * 2 * kH + 32 * t + m;
      npb[t] = -(p[0] + be[t]);
      nqb[t] = -(p[kH] + be[t]);
      dai[t] = a.dA[(int64_t)i * a.ldda + 32 * t + m];
      dq[t] = 0.f;
      cnt[t] = 0.f;
    }
    for (int64_t eb = e0; eb < e1; eb += 32) {
      const EdgeRows x = edge_rows(a, eb, e1, m, kh);
      const int lim = (int)(e1 - eb);  // rows below lim are edges of node i
      float xt[16];
      unsigned poff[16], doff[16];
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int row = mr0 + 8 * (r >> 2) + (r & 3);
        const unsigned j = (unsigned)__shfl(x.j, row);
        poff[r] = j * (2 * kH * 4) + 4 * m;
        doff[r] = j * dpitch + 4 * m;
        xt[r] = a.E[(eb + (row < lim ? row : lim - 1)) * kE + fk];
      }
      const float xs[8] = {x.x0.x, x.x0.y, x.x0.z, x.x0.w, x.x1.x, x.x1.y, x.x1.z, x.x1.w};
      bf16x8 ah, am, al, f1[2], f2[2];
#pragma unroll
      for (int s = 0; s < 8; ++s) {
        __bf16 h, md, l;
        split3_bf16(xs[s], h, md, l);
        if (s == kPastSlot - 8 && kh) h = (__bf16)(m < lim ? 0.f : 1.f);
        ah[s] = h;
        am[s] = md;
        al[s] = l;
      }
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        __bf16 h, md, l;
        split3_bf16(m == kPastSlot ? 1.f : xt[r], h, md, l);
        f1[r >> 3][r & 7] = m < 16 ? h : md;
        f2[r >> 3][r & 7] = m < 16 ? l : (__bf16)0.f;
      }
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        f32x16 zs, zt;
        float d[16];
#pragma unroll
        for (int r = 0; r < 16; ++r) zt[r] = *(const float*)(Pb + 128 * t + poff[r]);
#pragma unroll
        for (int r = 0; r < 16; ++r) zs[r] = *(const float*)(Pb + kH * 4 + 128 * t + poff[r]);
#pragma unroll
        for (int r = 0; r < 16; ++r) d[r] = *(const float*)(Db + 128 * t + doff[r]);
        __builtin_amdgcn_sched_barrier(0);
        const bf16x8* w = wfrag + t * 64 + lane;
        zt = edge_product(ah, am, al, w + 3 * 256, zt);
        zs = edge_product(ah, am, al, w, zs);
        float q0 = 0.f, q1 = 0.f;
#pragma unroll
        for (int r = 0; r < 16; r += 2) {
          q0 += zt[r] > nqb[t] ? d[r] : 0.f;
          q1 += zt[r + 1] > nqb[t] ? d[r + 1] : 0.f;
        }
        dq[t] += q0 + q1;
        bf16x8 mk[2];
#pragma unroll
        for (int r = 0; r < 16; ++r)
          mk[r >> 3][r & 7] = (__bf16)(zs[r] > npb[t] ? 1.f : 0.f);
        f32x16 g = {};
        g = __builtin_amdgcn_mfma_f32_32x32x16_bf16(f2[0], mk[0], g, 0, 0, 0);
        g = __builtin_amdgcn_mfma_f32_32x32x16_bf16(f2[1], mk[1], g, 0, 0, 0);
        g = __builtin_amdgcn_mfma_f32_32x32x16_bf16(f1[0], mk[0], g, 0, 0, 0);
        g = __builtin_amdgcn_mfma_f32_32x32x16_bf16(f1[1], mk[1], g, 0, 0, 0);
        cnt[t] += g[5];  // row 13 in the upper half-wave
#pragma unroll
        for (int r = 0; r < 8; ++r) gt[t][r] = fmaf(dai[t], g[r] + g[8 + r], gt[t][r]);
        hold_order(dq[t]);
      }
    }
    // the lower half-wave stores dQ, the upper one dP
    __bf16* const o = a.dPQb + (int64_t)i * 2 * kH + (hf ? 0 : kH) + m;
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      const float q = dq[t] + __shfl_xor(dq[t], 32);
      o[32 * t] = (__bf16)(hf ? cnt[t] * dai[t] : q);
    }
  }
  // the block's sum in wave order
  for (int w = 0; w < 4; ++w) {
    if (w == wv) {
#pragma unroll
      for (int t = 0; t < 4; ++t)
#pragma unroll
        for (int r = 0; r < 8; ++r) {
          const int k = 8 * (r >> 2) + mr0 + (r & 3), c = 32 * t + m;
          if (k == kPastSlot)
            slab[kE * kH + c] += gt[t][r];
          else
            slab[k * kH + c] += gt[t][r];
        }
    }
    __syncthreads();
  }
  float* p = a.part + (int64_t)blockIdx.x * (kE + 1) * kH;
  for (int f = threadIdx.x; f < (kE + 1) * kH; f += 256) p[f] = slab[f];
}

// ---------------------------------------------------------------------------
// decoder, loss, elementwise pieces
// ---------------------------------------------------------------------------
// Y = H W_out + b_out + the node's SPH pressure and viscosity
// accelerations / g (FP32 skip path; one thread per node).
__global__ __launch_bounds__(256) void decode_kernel(int n, const float* __restrict__ H,
                                                     const float* __restrict__ W,
                                                     const float* __restrict__ b,
                                                     const float* __restrict__ acc4,
                                                     float* __restrict__ Y) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i >= n) return;
  const float* a4 = acc4 + (int64_t)i * 4;
  float y0 = b[0] + a4[0] + a4[2], y1 = b[1] + a4[1] + a4[3];
  const float* h = H + (int64_t)i * kH;
  for (int c = 0; c < kH; ++c) {
    const float v = h[c];
    y0 += v * W[c * kOut];
    y1 += v * W[c * kOut + 1];
  }
  Y[2 * (int64_t)i] = y0;
  Y[2 * (int64_t)i + 1] = y1;
}

// dH = dY W_out^T; per-block (64 nodes) partials of dW_out = H^T dY and db_out.
__global__ __launch_bounds__(256) void decode_bwd_kernel(int n, const float* __restrict__ H,
                                                         const float* __restrict__ W,
                                                         const float* __restrict__ dY,
                                                         float* __restrict__ dH,
                                                         float* __restrict__ part) {
  __shared__ float sw[2][256];
  __shared__ float sb[2][64];
  const int node0 = blockIdx.x * 64;
  const int t = threadIdx.x;
  const int c = t & (kH - 1);
  const int half = t >> 7;
  const float w0 = W[c * kOut], w1 = W[c * kOut + 1];
  float gw0 = 0.f, gw1 = 0.f;
  for (int k = half; k < 64; k += 2) {
    const int i = node0 + k;
    if (i >= n) break;
    const float d0 = dY[2 * (int64_t)i], d1 = dY[2 * (int64_t)i + 1];
    dH[(int64_t)i * kH + c] = d0 * w0 + d1 * w1;
    const float h = H[(int64_t)i * kH + c];
    gw0 += h * d0;
    gw1 += h * d1;
  }
  sw[0][t] = gw0;
  sw[1][t] = gw1;
  if (t < 64) {
    const int i = node0 + t;
    sb[0][t] = i < n ? dY[2 * (int64_t)i] : 0.f;
    sb[1][t] = i < n ? dY[2 * (int64_t)i + 1] : 0.f;
  }
  __syncthreads();
  float* p = part + (int64_t)blockIdx.x * (kH * kOut + kOut);
  if (t < kH) {
    p[t * kOut] = sw[0][t] + sw[0][t + kH];
    p[t * kOut + 1] = sw[1][t] + sw[1][t + kH];
  }
  if (t == 0) {
    float s0 = 0.f, s1 = 0.f;
    for (int k = 0; k < 64; ++k) {
      s0 += sb[0][k];
      s1 += sb[1][k];
    }
    p[kH * kOut] = s0;
    p[kH * kOut + 1] = s1;
  }
}

// MSE over fluid nodes of (Y - T): per-block partial losses and dY.
__global__ __launch_bounds__(256) void loss_kernel(int n, const int* __restrict__ btype,
                                                   const float* __restrict__ Y,
                                                   const float* __restrict__ T, float inv_nf,
                                                   float* __restrict__ dY,
                                                   float* __restrict__ part) {
  __shared__ float red[256];
  const int i = blockIdx.x * 256 + threadIdx.x;
  float l = 0.f;
  if (i < n) {
    const bool fl = btype[i] == 0;
    const float e0 = fl ? Y[2 * (int64_t)i] - T[2 * (int64_t)i] : 0.f;
    const float e1 = fl ? Y[2 * (int64_t)i + 1] - T[2 * (int64_t)i + 1] : 0.f;
    l = (e0 * e0 + e1 * e1) * inv_nf;
    dY[2 * (int64_t)i] = 2.f * e0 * inv_nf;
    dY[2 * (int64_t)i + 1] = 2.f * e1 * inv_nf;
  }
  red[threadIdx.x] = l;
  __syncthreads();
  for (int s = 128; s > 0; s >>= 1) {
    if (threadIdx.x < s) red[threadIdx.x] += red[threadIdx.x + s];
    __syncthreads();
  }
  if (threadIdx.x == 0) part[blockIdx.x] = red[0];
}

// outb = BF16(mask(act > 0) * d) and, per block of kReluRows rows, the column
// sums of the masked FP32 values (the bias gradient's partials): nothing else
// reads the FP32 values, so they are not stored.  32 lanes x 4 columns cover
// a row of kH, eight rows at a time.  (Masking and summing in launches of
// their own took 16 + 61 us for 33k rows; this one 9 us.)
constexpr int kReluRows = 64;
__global__ __launch_bounds__(256) void relu_bwd_kernel(int rows, const float* __restrict__ act,
                                                       const float* __restrict__ d,
                                                       __bf16* __restrict__ outb,
                                                       float* __restrict__ part) {
  __shared__ float4 red[8][32];
  typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
  const int c = threadIdx.x & 31, k = threadIdx.x >> 5;
  const int r0 = blockIdx.x * kReluRows;
  float4 s = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
  for (int i = 0; i < kReluRows / 8; ++i) {
    const int r = r0 + 8 * i + k;
    if (r >= rows) break;
    const int64_t o = (int64_t)r * kH + 4 * c;
    const float4 a = *(const float4*)(act + o);
    const float4 v = *(const float4*)(d + o);
    const float4 z = make_float4(a.x > 0.f ? v.x : 0.f, a.y > 0.f ? v.y : 0.f,
                                 a.z > 0.f ? v.z : 0.f, a.w > 0.f ? v.w : 0.f);
    const bf16x4 zb = {(__bf16)z.x, (__bf16)z.y, (__bf16)z.z, (__bf16)z.w};
    *(bf16x4*)(outb + o) = zb;
    s.x += z.x;
    s.y += z.y;
    s.z += z.z;
    s.w += z.w;
  }
  red[k][c] = s;
  __syncthreads();
  if (threadIdx.x < kH) {
    const int col = threadIdx.x;
    float t = 0.f;
#pragma unroll
    for (int i = 0; i < 8; ++i) t += ((const float*)red[i])[col];
    part[(int64_t)blockIdx.x * kH + col] = t;
  }
}

__global__ __launch_bounds__(256) void adam_kernel(int64_t n, float* __restrict__ w,
                                                   __bf16* __restrict__ wb,
                                                   const float* __restrict__ g,
                                                   float* __restrict__ m, float* __restrict__ v,
                                                   float lr, float b1, float b2, float eps,
                                                   float c1, float c2) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= n) return;
  const float gi = g[i];
  const float mi = b1 * m[i] + (1.f - b1) * gi;
  const float vi = b2 * v[i] + (1.f - b2) * gi * gi;
  m[i] = mi;
  v[i] = vi;
  const float wi = w[i] - lr * (mi / c1) / (sqrtf(vi / c2) + eps);
  w[i] = wi;
  wb[i] = (__bf16)wi;
}

__global__ __launch_bounds__(256) void to_bf16_kernel(int64_t n, const float* __restrict__ w,
                                                      __bf16* __restrict__ wb) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i < n) wb[i] = (__bf16)w[i];
}

__global__ __launch_bounds__(256) void fill_f32_kernel(int64_t n, float* __restrict__ p,
                                                       float v) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i < n) p[i] = v;
}

// Surrogate update of fluid nodes (symplectic Euler): u += dt a g, x += dt u.
__global__ __launch_bounds__(256) void integrate_kernel(int64_t n, const int* __restrict__ btype,
                                                        const float* __restrict__ Y, float ag,
                                                        float dt, float* __restrict__ x,
                                                        float* __restrict__ y,
                                                        float* __restrict__ u,
                                                        float* __restrict__ v) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= n || btype[i] != 0) return;
  const float u1 = u[i] + dt * ag * Y[2 * i];
  const float v1 = v[i] + dt * ag * Y[2 * i + 1];
  u[i] = u1;
  v[i] = v1;
  x[i] = x[i] + dt * u1;
  y[i] = y[i] + dt * v1;
}

// ---------------------------------------------------------------------------
// model object
// ---------------------------------------------------------------------------
struct Buf {
  void* p = nullptr;
  size_t bytes = 0;
};

struct Model {
  Layout L;
  float* w = nullptr;     // FP32 master
  __bf16* wb = nullptr;   // BF16 copy
  __bf16* wbt = nullptr;  // BF16 copies of the GEMM weights, transposed
  float* g = nullptr;     // gradients
  float* m = nullptr;     // Adam moments
  float* v = nullptr;
  // activations and scratch, grown on demand
  // optional per-category launch timing of the forward pass: features,
  // GEMMs, edge aggregation, decoder
  int timing = 0;
  double t_ms[4] = {0, 0, 0, 0};
  int64_t t_calls = 0;
  std::vector<hipEvent_t> ev;
  Buf X, E, N4, H[kR + 1], HA[kR], PQ[kR], U[kR], dH, dZb, dA, dPQb, part, lossp;
  int64_t n_act = -1, e_act = -1;
  bool acts = false;  // the last forward pass stored what the backward pass reads
};

// Events around each launch of a timed forward pass.
struct Timer {
  Model* M;
  hipStream_t st;
  std::vector<std::pair<int, int>> marks;  // (category, event index of the start)
  int used = 0;
  Timer(Model* m, hipStream_t s) : M(m), st(s) {}
  void begin(int cat) {
    if (!M->timing) return;
    while ((int)M->ev.size() < used + 2) {
      hipEvent_t e;
      if (hipEventCreate(&e) != hipSuccess) {
        M->timing = 0;
        return;
      }
      M->ev.push_back(e);
    }
    (void)hipEventRecord(M->ev[used], st);
    marks.push_back({cat, used});
    used += 2;
  }
  void end() {
    if (!M->timing || marks.empty()) return;
    (void)hipEventRecord(M->ev[marks.back().second + 1], st);
  }
  void collect() {
    if (!M->timing || marks.empty()) return;
    (void)hipEventSynchronize(M->ev[marks.back().second + 1]);
    for (auto& m : marks) {
      float ms = 0.f;
      if (hipEventElapsedTime(&ms, M->ev[m.second], M->ev[m.second + 1]) == hipSuccess)
        M->t_ms[m.first] += ms;
    }
    M->t_calls += 1;
  }
};

static int32_t ensure(Buf& b, size_t bytes) {
  if (b.bytes >= bytes && b.p) return SPH_OK;
  if (b.p) {
    // earlier launches may still read the old buffer
    (void)hipDeviceSynchronize();
    (void)hipFree(b.p);
  }
  b.p = nullptr;
  b.bytes = 0;
  hipError_t e = hipMalloc(&b.p, bytes < 256 ? 256 : bytes);
  if (e != hipSuccess) {
    set_error("sph_mlp: allocation of %zu bytes: %s", bytes, hipGetErrorString(e));
    return (int32_t)e;
  }
  b.bytes = bytes;
  return SPH_OK;
}

static int nblk(int64_t n) { return (int)((n + 255) / 256); }

// Persistent edge aggregation: up to SPH_EDGE_WAVES waves per SIMD of the
// 256 CUs; a block's four waves take the nodes of its run (node_run) in turn.
static int edge_fwd_blocks(int64_t n) {
  const int64_t waves = std::min<int64_t>(n, 256 * 4 * SPH_EDGE_WAVES);
  return (int)std::max<int64_t>(1, (waves + 3) / 4);
}

static int32_t gemm(hipStream_t st, const GemmArgs& a) {
  dim3 grid((a.N + 63) / 64, (a.M + 63) / 64, 1);
  if (a.K == 16) {
    hipLaunchKernelGGL(gemm_nt16_kernel, grid, dim3(256), 0, st, a);
  } else if (a.K == 128 && a.C2 != nullptr) {
    hipLaunchKernelGGL((gemm_nt_lds_kernel<8, true>), grid, dim3(256), 0, st, a);
  } else if (a.K == 128) {
    hipLaunchKernelGGL(gemm_nt_lds_kernel<8>, grid, dim3(256), 0, st, a);
  } else if (a.K == 256) {
    hipLaunchKernelGGL(gemm_nt_lds_kernel<16>, grid, dim3(256), 0, st, a);
  } else {
    set_error("sph_mlp: no product of depth %d", a.K);
    return SPH_EUNSUPPORTED;
  }
  return launch_status("sph_mlp/gemm");
}

static GemmArgs gargs(int M, int N, int K, const __bf16* A, int64_t lda, const __bf16* B,
                      int64_t ldb) {
  GemmArgs a{};
  a.M = M;
  a.N = N;
  a.K = K;
  a.A = A;
  a.lda = lda;
  a.B = B;
  a.ldb = ldb;
  return a;
}

// Row chunks of a weight gradient: at most 256 rows each while that makes up
// to 64 of them, enough blocks for the 256 CUs (four tiles of 128 x 64 per
// matrix), longer ones after that: a slab's 128 KB of output stays small
// against the rows it reads.
static int grad_splits(int rows) { return std::max(1, std::min(64, (rows + 255) / 256)); }

// Weight gradient G[kdim x ncols] += X^T D with X [rows x kdim] (ldx), D
// [rows x ncols] (ldd): a slab per chunk of rows, then the fixed-order sum.
static int32_t weight_grad(Model* M, hipStream_t st, int rows, int kdim, int ncols,
                           const __bf16* X, int64_t ldx, const __bf16* D, int64_t ldd,
                           float* G) {
  GradArgs a{};
  a.rows = rows;
  a.kdim = kdim;
  a.ncols = ncols;
  a.X = X;
  a.ldx = ldx;
  a.D = D;
  a.ldd = ldd;
  const int splits = grad_splits(rows);
  a.chunk = ((rows + splits - 1) / splits + 31) / 32 * 32;
  const int nz = (rows + a.chunk - 1) / a.chunk;
  const int64_t slab = (int64_t)kdim * ncols;
  SPH_TRY(ensure(M->part, (size_t)nz * slab * 4 + 1024));
  a.part = (float*)M->part.p;
  if (kdim <= 32)
    hipLaunchKernelGGL((grad_kernel<32, 128>), dim3((ncols + 127) / 128, 1, nz), dim3(256), 0, st,
                       a);
  else
    hipLaunchKernelGGL((grad_kernel<128, 64>), dim3((ncols + 63) / 64, (kdim + 127) / 128, nz),
                       dim3(256), 0, st, a);
  slab_sum(st, (const float*)M->part.p, nz, slab, (int)slab, G, 1);
  return launch_status("sph_mlp/weight_grad");
}

// dZb = BF16(d masked by act > 0) and the bias gradient G[kH] += its column
// sums.
static int32_t relu_bias_grad(Model* M, hipStream_t st, int rows, const float* act,
                              const float* d, __bf16* dZb, float* G) {
  const int nb = (rows + kReluRows - 1) / kReluRows;
  SPH_TRY(ensure(M->part, (size_t)nb * kH * 4 + 1024));
  hipLaunchKernelGGL(relu_bwd_kernel, dim3(nb), dim3(256), 0, st, rows, act, d, dZb,
                     (float*)M->part.p);
  slab_sum(st, (const float*)M->part.p, nb, kH, kH, G, 1);
  return launch_status("sph_mlp/relu_bwd");
}

static FeatArgs feat_args(const sph_mlp_graph* g) {
  FeatArgs f;
  f.n = (int)g->n;
  f.pos4 = (const float4*)g->pos4;
  f.vel4 = (const float4*)g->vel4;
  f.rho = g->rho;
  f.btype = g->btype;
  f.off = g->off;
  f.nbr = g->nbr;
  f.ne = g->nedges;
  f.rho0 = (float)g->rho0;
  f.co = (float)g->co;
  f.gamma = (float)g->gamma;
  f.B = (float)(g->co * g->co * g->rho0 / g->gamma);
  f.u_scale = (float)g->u_scale;
  f.g = (float)g->g;
  f.rho_scale = (float)g->rho_scale;
  f.alpha = (float)g->alpha;
  f.eta = (float)g->eta;
  f.dim = g->dim;
  return f;
}

static int32_t check_graph(const sph_mlp_graph* g, const char* who) {
  if (!g || g->n < 0 || g->n > INT32_MAX / 4 || g->nedges < 0 ||
      (g->n > 0 && (!g->pos4 || !g->vel4 || !g->rho || !g->btype || !g->off || !g->nbr)) ||
      !(g->rho0 > 0) || !(g->u_scale > 0) || !(g->g > 0) || (g->dim != 2 && g->dim != 3)) {
    set_error("%s: invalid graph", who);
    return SPH_EINVAL;
  }
  return SPH_OK;
}

// Transposed BF16 copies of the GEMM weights (W_in, W_ab, W_u).
static int32_t refresh_transposed(Model* M, hipStream_t st) {
  const Layout& L = M->L;
  struct Mat {
    int64_t off;
    int K, N;
  };
  std::vector<Mat> mats = {{L.w_in, kIn, kH}};
  for (int r = 0; r < kR; ++r) {
    mats.push_back({L.w_ab[r], kH, 2 * kH});
    mats.push_back({L.w_u[r], 2 * kH, kH});
  }
  for (const Mat& m : mats)
    hipLaunchKernelGGL(transpose_bf16_kernel, dim3(nblk((int64_t)m.K * m.N)), dim3(256), 0, st,
                       m.K, m.N, M->w + m.off, M->wbt + m.off);
  return launch_status("sph_mlp/transpose");
}

}  // namespace mlp
}  // namespace sph

using namespace sph;
using namespace sph::mlp;

extern "C" {

int64_t sph_mlp_param_count(void) { return layout().total; }

int32_t sph_mlp_create(void** model) {
  if (!model) {
    set_error("sph_mlp_create: NULL output");
    return SPH_EINVAL;
  }
  Model* M = new Model();
  M->L = layout();
  const size_t n = (size_t)M->L.total;
  hipError_t e = hipMalloc((void**)&M->w, n * 4);
  if (e == hipSuccess) e = hipMalloc((void**)&M->wb, n * 2);
  if (e == hipSuccess) e = hipMalloc((void**)&M->wbt, n * 2);
  if (e == hipSuccess) e = hipMalloc((void**)&M->g, n * 4);
  if (e == hipSuccess) e = hipMalloc((void**)&M->m, n * 4);
  if (e == hipSuccess) e = hipMalloc((void**)&M->v, n * 4);
  if (e == hipSuccess) e = hipMemset(M->w, 0, n * 4);
  if (e == hipSuccess) e = hipMemset(M->wb, 0, n * 2);
  if (e == hipSuccess) e = hipMemset(M->g, 0, n * 4);
  if (e == hipSuccess) e = hipMemset(M->m, 0, n * 4);
  if (e == hipSuccess) e = hipMemset(M->v, 0, n * 4);
  if (e != hipSuccess) {
    set_error("sph_mlp_create: %s", hipGetErrorString(e));
    return (int32_t)e;
  }
  *model = M;
  return SPH_OK;
}

int32_t sph_mlp_destroy(void* model) {
  Model* M = (Model*)model;
  if (!M) return SPH_OK;
  for (void* p : {(void*)M->w, (void*)M->wb, (void*)M->wbt, (void*)M->g, (void*)M->m,
                  (void*)M->v})
    (void)hipFree(p);
  for (hipEvent_t e : M->ev) (void)hipEventDestroy(e);
  for (Buf* b : {&M->X, &M->E, &M->N4, &M->dH, &M->dZb, &M->dA, &M->dPQb, &M->part,
                 &M->lossp})
    (void)hipFree(b->p);
  for (int r = 0; r <= kR; ++r) (void)hipFree(M->H[r].p);
  for (int r = 0; r < kR; ++r) {
    (void)hipFree(M->HA[r].p);
    (void)hipFree(M->PQ[r].p);
    (void)hipFree(M->U[r].p);
  }
  delete M;
  return SPH_OK;
}

// Synchronous copies of all parameters / gradients (FP32, layout order).
int32_t sph_mlp_set_params(void* model, const float* host) {
  Model* M = (Model*)model;
  if (!M || !host) {
    set_error("sph_mlp_set_params: bad arguments");
    return SPH_EINVAL;
  }
  hipError_t e = hipMemcpy(M->w, host, M->L.total * 4, hipMemcpyHostToDevice);
  if (e != hipSuccess) {
    set_error("sph_mlp_set_params: %s", hipGetErrorString(e));
    return (int32_t)e;
  }
  hipLaunchKernelGGL(to_bf16_kernel, dim3(nblk(M->L.total)), dim3(256), 0, 0, M->L.total, M->w,
                     M->wb);
  SPH_TRY(refresh_transposed(M, 0));
  e = hipDeviceSynchronize();
  if (e != hipSuccess) {
    set_error("sph_mlp_set_params: %s", hipGetErrorString(e));
    return (int32_t)e;
  }
  return SPH_OK;
}

int32_t sph_mlp_get(void* model, int32_t which, float* host) {
  Model* M = (Model*)model;
  if (!M || !host || which < 0 || which > 1) {
    set_error("sph_mlp_get: bad arguments");
    return SPH_EINVAL;
  }
  hipError_t e = hipDeviceSynchronize();
  if (e == hipSuccess)
    e = hipMemcpy(host, which == 0 ? M->w : M->g, M->L.total * 4, hipMemcpyDeviceToHost);
  if (e != hipSuccess) {
    set_error("sph_mlp_get: %s", hipGetErrorString(e));
    return (int32_t)e;
  }
  return SPH_OK;
}

int32_t sph_mlp_timing(void* model, int32_t enable, double* ms_host, int64_t* calls_host) {
  Model* M = (Model*)model;
  if (!M) {
    set_error("sph_mlp_timing: NULL model");
    return SPH_EINVAL;
  }
  if (ms_host)
    for (int k = 0; k < 4; ++k) ms_host[k] = M->t_ms[k];
  if (calls_host) *calls_host = M->t_calls;
  if (enable >= 0) {
    M->timing = enable ? 1 : 0;
    for (int k = 0; k < 4; ++k) M->t_ms[k] = 0.0;
    M->t_calls = 0;
  }
  return SPH_OK;
}

int32_t sph_mlp_zero_grad(void* model, void* stream) {
  Model* M = (Model*)model;
  if (!M) {
    set_error("sph_mlp_zero_grad: NULL model");
    return SPH_EINVAL;
  }
  hipLaunchKernelGGL(fill_f32_kernel, dim3(nblk(M->L.total)), dim3(256), 0, as_stream(stream),
                     M->L.total, M->g, 0.f);
  return launch_status("sph_mlp_zero_grad");
}

int32_t sph_mlp_forward(void* model, void* stream, const sph_mlp_graph* gr, float* out_dev) {
  Model* M = (Model*)model;
  if (!M || !out_dev) {
    set_error("sph_mlp_forward: bad arguments");
    return SPH_EINVAL;
  }
  SPH_TRY(check_graph(gr, "sph_mlp_forward"));
  const int64_t n = gr->n, ne = gr->nedges;
  if (n == 0) return SPH_OK;
  hipStream_t st = as_stream(stream);
  const Layout& L = M->L;
  SPH_TRY(ensure(M->X, (size_t)n * kIn * 2));
  SPH_TRY(ensure(M->E, (size_t)std::max<int64_t>(ne, 1) * kE * 4));
  for (int r = 0; r <= kR; ++r) SPH_TRY(ensure(M->H[r], (size_t)n * kH * 4));
  for (int r = 0; r < kR; ++r) {
    SPH_TRY(ensure(M->HA[r], (size_t)n * 2 * kH * 2));
    SPH_TRY(ensure(M->PQ[r], (size_t)n * 2 * kH * 4));
    SPH_TRY(ensure(M->U[r], (size_t)n * kH * 4));
  }
  M->n_act = n;
  M->e_act = ne;
  // inference: the pre-residual activations (the backward pass's ReLU
  // masks) are not stored
  const bool infer = (gr->flags & SPH_MLP_INFER) != 0;
  M->acts = !infer;
  SPH_TRY(ensure(M->N4, (size_t)n * 4 * 4));
  Timer T(M, st);
  const FeatArgs f = feat_args(gr);
  T.begin(0);
  hipLaunchKernelGGL(edge_feat_kernel, dim3((int)((n + kFeatNodes - 1) / kFeatNodes)), dim3(256),
                     0, st, f,
                     (float*)M->E.p, (float*)M->N4.p);
  hipLaunchKernelGGL(node_feat_kernel, dim3(nblk(n)), dim3(256), 0, st, f,
                     (const float*)M->N4.p, (__bf16*)M->X.p);
  T.end();
  SPH_TRY(launch_status("sph_mlp_forward/features"));
  // encoder: H0 = ReLU(X W_in + b_in) -> H[0] (FP32), HA[0] left half (BF16)
  {
    GemmArgs a = gargs((int)n, kH, kIn, (const __bf16*)M->X.p, kIn, M->wbt + L.w_in, kIn);
    a.C = (float*)M->H[0].p;
    a.ldc = kH;
    a.bias = M->w + L.b_in;
    a.relu = 1;
    a.Cb = (__bf16*)M->HA[0].p;
    a.ldcb = 2 * kH;
    T.begin(1);
    SPH_TRY(gemm(st, a));
    T.end();
  }
  for (int r = 0; r < kR; ++r) {
    __bf16* HA = (__bf16*)M->HA[r].p;
    float* PQ = (float*)M->PQ[r].p;
    {  // [P | Q] = H W_ab
      GemmArgs a = gargs((int)n, 2 * kH, kH, HA, 2 * kH, M->wbt + L.w_ab[r], kH);
      a.C = PQ;
      a.ldc = 2 * kH;
      T.begin(1);
      SPH_TRY(gemm(st, a));
      T.end();
    }
    EdgeArgs e{};
    e.n = (int)n;
    e.off = gr->off;
    e.nbr = gr->nbr;
    e.ne = gr->nedges;
    e.E = (const float*)M->E.p;
    e.PQ = PQ;
    e.Wc = M->w + L.w_c[r];
    e.be = M->w + L.b_e[r];
    e.A = HA + kH;
    e.lda = 2 * kH;
    T.begin(2);
    // the MFMA kernel addresses Q rows by 32-bit byte offsets (n * 8 kH < 2^32)
    if (SPH_EDGE_MFMA && !(gr->flags & SPH_MLP_EDGE_FP32) && n < (int64_t(1) << 22))
      hipLaunchKernelGGL(edge_fwd_mfma_kernel, dim3(edge_fwd_blocks(n)), dim3(256), 0, st, e, e.off);
    else
      hipLaunchKernelGGL(edge_fwd_kernel, dim3((int)((n + 3) / 4)), dim3(256), 0, st, e);
    T.end();
    SPH_TRY(launch_status("sph_mlp_forward/edges"));
    {  // U = ReLU([H | A] W_u + c_u); H' = H + U
      GemmArgs a = gargs((int)n, kH, 2 * kH, HA, 2 * kH, M->wbt + L.w_u[r], 2 * kH);
      a.bias = M->w + L.c_u[r];
      a.relu = 1;
      a.U = infer ? nullptr : (float*)M->U[r].p;
      a.ldu = kH;
      a.res = (const float*)M->H[r].p;
      a.ldr = kH;
      a.C = (float*)M->H[r + 1].p;
      a.ldc = kH;
      if (r + 1 < kR) {
        a.Cb = (__bf16*)M->HA[r + 1].p;
        a.ldcb = 2 * kH;
      }
      T.begin(1);
      SPH_TRY(gemm(st, a));
      T.end();
    }
  }
  T.begin(3);
  hipLaunchKernelGGL(decode_kernel, dim3(nblk(n)), dim3(256), 0, st, (int)n,
                     (const float*)M->H[kR].p, M->w + L.w_out, M->w + L.b_out,
                     (const float*)M->N4.p, out_dev);
  T.end();
  SPH_TRY(launch_status("sph_mlp_forward"));
  T.collect();
  return SPH_OK;
}

int32_t sph_mlp_loss(void* model, void* stream, const sph_mlp_graph* gr, const float* out_dev,
                     const float* target_dev, float* loss_dev, float* dout_dev) {
  Model* M = (Model*)model;
  if (!M || !out_dev || !target_dev || !loss_dev || !dout_dev) {
    set_error("sph_mlp_loss: bad arguments");
    return SPH_EINVAL;
  }
  SPH_TRY(check_graph(gr, "sph_mlp_loss"));
  const int64_t n = gr->n;
  if (n == 0) return SPH_OK;
  hipStream_t st = as_stream(stream);
  const int nb = nblk(n);
  SPH_TRY(ensure(M->lossp, (size_t)nb * 4 + 256));
  const float inv_nf = gr->n_fluid > 0 ? 1.f / (float)gr->n_fluid : 0.f;
  hipLaunchKernelGGL(loss_kernel, dim3(nb), dim3(256), 0, st, (int)n, gr->btype, out_dev,
                     target_dev, inv_nf, dout_dev, (float*)M->lossp.p);
  slab_sum(st, (const float*)M->lossp.p, nb, 1, 1, loss_dev, 0);
  return launch_status("sph_mlp_loss");
}

int32_t sph_mlp_backward(void* model, void* stream, const sph_mlp_graph* gr,
                         const float* dout_dev) {
  Model* M = (Model*)model;
  if (!M || !dout_dev) {
    set_error("sph_mlp_backward: bad arguments");
    return SPH_EINVAL;
  }
  SPH_TRY(check_graph(gr, "sph_mlp_backward"));
  const int64_t n = gr->n;
  if (n == 0) return SPH_OK;
  if (M->n_act != n || M->e_act != gr->nedges || !M->acts) {
    set_error("sph_mlp_backward: needs the forward pass of the same graph first (without "
              "SPH_MLP_INFER)");
    return SPH_EINVAL;
  }
  hipStream_t st = as_stream(stream);
  const Layout& L = M->L;
  SPH_TRY(ensure(M->dH, (size_t)n * kH * 4));
  SPH_TRY(ensure(M->dZb, (size_t)n * kH * 2));
  SPH_TRY(ensure(M->dA, (size_t)n * kH * 4));
  SPH_TRY(ensure(M->dPQb, (size_t)n * 2 * kH * 2));
  {
    // one scratch buffer serves every partial reduction of this pass: size
    // it once, before any launch reads it
    const int64_t wg = 64LL * 2 * kH * kH;                       // weight-gradient slabs
    const int64_t eg = 1024LL * 4 * (kE + 1) * kH;                // edge partials
    const int64_t dg = ((n + 63) / 64) * (kH * kOut + kOut);      // decoder partials
    const int64_t bg = ((n + kReluRows - 1) / kReluRows) * kH;    // bias partials
    SPH_TRY(ensure(M->part, (size_t)std::max(std::max(wg, eg), std::max(dg, bg)) * 4 + 1024));
  }
  float* dH = (float*)M->dH.p;
  // decoder
  {
    const int nb = (int)((n + 63) / 64);
    const int64_t per = kH * kOut + kOut;
    SPH_TRY(ensure(M->part, (size_t)nb * per * 4 + 1024));
    hipLaunchKernelGGL(decode_bwd_kernel, dim3(nb), dim3(256), 0, st, (int)n,
                       (const float*)M->H[kR].p, M->w + L.w_out, dout_dev, dH,
                       (float*)M->part.p);
    // W_out and b_out are contiguous: one slab sum over blocks
    slab_sum(st, (const float*)M->part.p, nb, per, (int)per, M->g + L.w_out, 1);
    SPH_TRY(launch_status("sph_mlp_backward/decoder"));
  }
  for (int r = kR - 1; r >= 0; --r) {
    __bf16* dZb = (__bf16*)M->dZb.p;
    // dZ = dH' * (U > 0), dc_u
    SPH_TRY(relu_bias_grad(M, st, (int)n, (const float*)M->U[r].p, dH, dZb, M->g + L.c_u[r]));
    // dW_u += [H | A]^T dZ
    SPH_TRY(weight_grad(M, st, (int)n, 2 * kH, kH, (const __bf16*)M->HA[r].p, 2 * kH, dZb, kH,
                        M->g + L.w_u[r]));
    {  // d[H | A] = dZ W_u^T: dH_r = dH' + d[H], dA
      GemmArgs a = gargs((int)n, 2 * kH, kH, dZb, kH, M->wb + L.w_u[r], kH);
      a.C = dH;
      a.ldc = kH;
      a.accumulate = 1;
      a.C2 = (float*)M->dA.p;
      a.ldc2 = kH;
      a.n2 = kH;
      SPH_TRY(gemm(st, a));
    }
    // edges: dP, dQ, dWc, dbe
    EdgeArgs e{};
    e.n = (int)n;
    e.off = gr->off;
    e.nbr = gr->nbr;
    e.ne = gr->nedges;
    e.E = (const float*)M->E.p;
    e.PQ = (const float*)M->PQ[r].p;
    e.Wc = M->w + L.w_c[r];
    e.be = M->w + L.b_e[r];
    e.dA = (const float*)M->dA.p;
    e.ldda = kH;
    e.dPQb = (__bf16*)M->dPQb.p;
    // the matrix-core kernel addresses rows by 32-bit byte offsets, as in the
    // forward pass; one slab per block, else per wave
    const bool mfma = SPH_EDGE_MFMA && !(gr->flags & SPH_MLP_EDGE_FP32) && n < (int64_t(1) << 22);
    const int nbk = (int)std::min<int64_t>(mfma ? 256 * kBwdWaves : 1024, (n + 3) / 4);
    const int nslab = mfma ? nbk : nbk * 4;
    const int64_t per = (int64_t)(kE + 1) * kH;
    SPH_TRY(ensure(M->part, (size_t)nslab * per * 4 + 1024));
    e.part = (float*)M->part.p;
    if (mfma)
      hipLaunchKernelGGL(edge_bwd_mfma_kernel, dim3(nbk), dim3(256), 0, st, e, e.off);
    else
      hipLaunchKernelGGL(edge_bwd_kernel, dim3(nbk), dim3(256), 0, st, e);
    // W_c and b_e are contiguous
    slab_sum(st, (const float*)M->part.p, nslab, per, (int)per, M->g + L.w_c[r], 1);
    SPH_TRY(launch_status("sph_mlp_backward/edges"));
    // dW_ab += H^T dPQ
    SPH_TRY(weight_grad(M, st, (int)n, kH, 2 * kH, (const __bf16*)M->HA[r].p, 2 * kH,
                        (const __bf16*)M->dPQb.p, 2 * kH, M->g + L.w_ab[r]));
    {  // dH += dPQ W_ab^T
      GemmArgs a = gargs((int)n, kH, 2 * kH, (const __bf16*)M->dPQb.p, 2 * kH,
                         M->wb + L.w_ab[r], 2 * kH);
      a.C = dH;
      a.ldc = kH;
      a.accumulate = 1;
      SPH_TRY(gemm(st, a));
    }
  }
  // encoder: dZ0 = dH * (H0 > 0); dW_in += X^T dZ0; db_in
  {
    __bf16* dZb = (__bf16*)M->dZb.p;
    SPH_TRY(relu_bias_grad(M, st, (int)n, (const float*)M->H[0].p, dH, dZb, M->g + L.b_in));
    SPH_TRY(weight_grad(M, st, (int)n, kIn, kH, (const __bf16*)M->X.p, kIn, dZb, kH,
                        M->g + L.w_in));
  }
  return launch_status("sph_mlp_backward");
}

int32_t sph_mlp_adam(void* model, void* stream, float lr, float b1, float b2, float eps,
                     int32_t t) {
  Model* M = (Model*)model;
  if (!M || t < 1) {
    set_error("sph_mlp_adam: bad arguments");
    return SPH_EINVAL;
  }
  const float c1 = 1.f - powf(b1, (float)t), c2 = 1.f - powf(b2, (float)t);
  hipLaunchKernelGGL(adam_kernel, dim3(nblk(M->L.total)), dim3(256), 0, as_stream(stream),
                     M->L.total, M->w, M->wb, M->g, M->m, M->v, lr, b1, b2, eps, c1, c2);
  SPH_TRY(launch_status("sph_mlp_adam"));
  return refresh_transposed(M, as_stream(stream));
}

int32_t sph_mlp_integrate(void* stream, int64_t n, const int32_t* btype, const float* out_dev,
                          double a_scale, double dt, float* x, float* y, float* u, float* v) {
  if (n < 0 || (n > 0 && (!btype || !out_dev || !x || !y || !u || !v))) {
    set_error("sph_mlp_integrate: bad arguments");
    return SPH_EINVAL;
  }
  if (n == 0) return SPH_OK;
  hipLaunchKernelGGL(integrate_kernel, dim3(nblk(n)), dim3(256), 0, as_stream(stream), n, btype,
                     out_dev, (float)a_scale, (float)dt, x, y, u, v);
  return launch_status("sph_mlp_integrate");
}

}  // extern "C"
