/*
 * Learned large-step corrector: a message-passing graph network on the
 * Voronoi mesh that maps the state after one coarse large step (doubled dt,
 * fewer acoustic substeps) to the correction that brings it back onto the
 * fine-dt trajectory.  No reference counterpart: the reference dycore has no
 * learned component; the corrector sits after the reference's step boundary
 * (cuda_driver.py:5751 step_device) and the plain step is its fallback.
 *
 * Network (hidden width H = 128, NL message-passing layers):
 *   features  x_c = normalised column of 6 channels x 64 rows: the cell wind
 *             (U_east, U_north) by a least-squares fit of the normal
 *             velocities on edgesOnCell, w, theta_m, rho_zz, qv, plus the
 *             Coriolis parameter in a padding row                 [C][384]
 *   encoder   h0 = relu(x W_in + b_in)                           [C][128]
 *   layer l   a_c = mean_{j in cellsOnCell(c)} h_j
 *             h_{l+1} = h_l + relu([h_l, a] W_l + b_l)            [C][128]
 *   decoder   y = h_NL W_out + b_out                              [C][320]
 *             y = (dU_east, dU_north, dtheta_m, drho_zz, dw) x 64 rows
 *   edges     du_e = cos(a_e) (dU_east(c0)+dU_east(c1))/2
 *                  + sin(a_e) (dU_north(c0)+dU_north(c1))/2  (cellsOnEdge)
 * Every GEMM is a bf16 MFMA (v_mfma_f32_16x16x32_bf16) with fp32
 * accumulation; weights and activations are bf16, the Adam master weights,
 * moments and gradients fp32.  Weight gradients are reduced over cells in
 * per-block partials summed in a fixed order (repeatable bits).
 *
 * Loss: mean squared error of the normalised corrections of u (edges),
 * theta_m and rho_zz (cells) and w (interior interfaces), one mean per
 * variable, summed.
 */
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstring>
#include <string>
#include <vector>

#include "../../include/hexdyn.h"
#include "hexdyn_div.h"
#include "hexdyn_internal.h"

namespace hexdyn {
namespace net {
namespace {

typedef __bf16 bf16;
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

constexpr int HID = 128;
constexpr int KIN = 6 * HX_ROW;    // 384 input features per cell
constexpr int NOUT = 5 * HX_ROW;   // 320 outputs per cell
enum { CH_UE = 0, CH_UN = 1, CH_W = 2, CH_TH = 3, CH_RHO = 4, CH_QV = 5 };
enum { O_UE = 0, O_UN = 1, O_TH = 2, O_RHO = 3, O_W = 4 };

__device__ __forceinline__ f32x4 mfma(const bf16x8 &a, const bf16x8 &b, const f32x4 &c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}

// Logical block of a launch: XCD x (hardware block b runs on XCD b % 8) takes
// a contiguous range of the curve, so the rows its gathers share meet in its L2.
__device__ __forceinline__ int curve_block() {
  const int nb = (int)gridDim.x, b = (int)blockIdx.x;
  const int x = b & 7, i = b >> 3, q = nb >> 3, r = nb & 7;
  return (x < r) ? x * (q + 1) + i : r * (q + 1) + (x - r) * q + i;
}

// ------------------------------------------------------------------ GEMM
// out[M][N] = epi(A[M][K] . B), A row-major bf16, B given transposed
// (Bt[N][K], bf16).  A wavefront takes 16 rows at a time with every column of
// the block's NC: all K/32 fragments of A are requested before the block's
// copy of Bt (its NC rows) is staged in LDS, so one memory latency covers
// both, and 16 rows per wavefront keep every CU busy down to a few thousand
// rows (32 rows per wavefront and 8 wavefronts per block left 41 blocks at
// 10 242 rows: 30 us for a layer and its mean in two passes, 17 us here).
// The weights are the first MFMA operand and the rows of A the second: the
// accumulator lane l then holds row l % 16 of the tile and 4 consecutive
// columns 4 * (l / 16) + i, which store as 8 or 16 bytes (the other way round
// they are 4 rows of one column, 2 or 4 bytes each).  Operand layout
// (16x16x32): lane l supplies row l % 16 and the 8 consecutive k values
// 8 * (l / 16) .. +7.
// NE > 0: a message-passing layer.  A = [h_c | mean over cellsOnCell of h],
// the mean formed here from the neighbours' rows (fp32 sums in slot order, one
// rounding to bf16) instead of in a pass of its own.
enum { EPI_RELU = 0, EPI_RESID_RELU = 1, EPI_F32 = 2, EPI_F32_MASK = 3 };

struct GemmArgs {
  const bf16 *A, *Bt;
  const float *bias;
  const bf16 *resid;      // EPI_RESID_RELU: added after the relu
  const bf16 *mask;       // EPI_F32_MASK: out_b = out_f where mask > 0
  bf16 *out_b;
  float *out_f;
  bf16 *relu_out;         // EPI_RESID_RELU: the relu itself (kept for backward), may be null
  bf16 *mean_out;         // NE > 0: the neighbour mean (kept for backward), may be null
  const int *coc, *neoc;  // NE > 0
  int M;
};

typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));

template <int K, int NE>
__device__ __forceinline__ void gemm_rows(const GemmArgs &g, int tile, int lr, int lg, bf16x8 (&a)[K / 32]) {
  const int row = min(tile * 16 + lr, g.M - 1);
  constexpr int KO = NE > 0 ? K / 2 : K;  // the row's own columns
  const bf16 *own = g.A + (size_t)row * KO + lg * 8;
#pragma unroll
  for (int q = 0; q < KO / 32; ++q) a[q] = *(const bf16x8 *)(own + q * 32);
  if constexpr (NE > 0) {
    constexpr int Q = KO / 32, QH = Q / 2;
    const int n = g.neoc[row];
    int nb[NE];
#pragma unroll
    for (int s = 0; s < NE; ++s) nb[s] = g.coc[row * NE + s];  // padded slots hold cell 0
    const float fn = (float)n, rn = 1.0f / fn;
#pragma unroll
    for (int h = 0; h < 2; ++h) {  // half the channels at a time: every neighbour's row of them in flight together
      bf16x8 v[NE][QH];
#pragma unroll
      for (int s = 0; s < NE; ++s)
#pragma unroll
        for (int q = 0; q < QH; ++q)
          v[s][q] = *(const bf16x8 *)(g.A + (size_t)nb[s] * KO + (h * QH + q) * 32 + lg * 8);
#pragma unroll
      for (int q = 0; q < QH; ++q) {
        bf16x8 m;
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          float acc = 0.f;
#pragma unroll
          for (int s = 0; s < NE; ++s) acc = s < n ? acc + (float)v[s][q][j] : acc;
          m[j] = (bf16)div_count(acc, fn, rn);
        }
        a[Q + h * QH + q] = m;
        if (g.mean_out && tile * 16 + lr < g.M)
          *(bf16x8 *)(g.mean_out + (size_t)row * KO + (h * QH + q) * 32 + lg * 8) = m;
      }
    }
  }
}

template <int K, int N, int NC, int EPI, int NE>
__global__ void __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(4))) k_gemm(const GemmArgs g) {
  static_assert(K % 32 == 0 && NC % 16 == 0 && N % NC == 0, "tile shape");
  static_assert(NE == 0 || NC == N, "one block forms a row's neighbour mean");
  constexpr int LDK = K + 8;  // row stride in LDS (16-byte pad against bank conflicts)
  constexpr int NT = NC / 16;
  extern __shared__ __align__(16) unsigned char lds_raw[];
  bf16 *sB = (bf16 *)lds_raw;
  const int W = (int)(blockDim.x >> 6);
  const int w = (int)(threadIdx.x >> 6), l = (int)(threadIdx.x & 63);
  const int lr = l & 15, lg = l >> 4;
  const int n0 = (int)blockIdx.y * NC;
  const int tiles = (g.M + 15) / 16;
  int t = curve_block() * W + w;
  bf16x8 a[K / 32];
  if (t < tiles) gemm_rows<K, NE>(g, t, lr, lg, a);
  for (int i = (int)threadIdx.x; i < NC * (K / 8); i += 64 * W) {
    const int n = i / (K / 8), kc = i % (K / 8);
    *(bf16x8 *)(sB + n * LDK + kc * 8) = *(const bf16x8 *)(g.Bt + (size_t)(n0 + n) * K + kc * 8);
  }
  __syncthreads();
  while (t < tiles) {
    asm volatile("" ::: "memory");  // the fragments of B are read from LDS per tile, not kept across tiles
    f32x4 acc[NT];
#pragma unroll
    for (int j = 0; j < NT; ++j) acc[j] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int q = 0; q < K / 32; ++q)
#pragma unroll
      for (int j = 0; j < NT; ++j) {
        const bf16x8 b = *(const bf16x8 *)(sB + (j * 16 + lr) * LDK + q * 32 + lg * 8);
        acc[j] = mfma(b, a[q], acc[j]);
      }
    const int row = t * 16 + lr;
    if (row < g.M) {
#pragma unroll
      for (int j = 0; j < NT; ++j) {
        const int col = n0 + j * 16 + lg * 4;
        const size_t o = (size_t)row * N + col;
        f32x4 v = acc[j];
        if (g.bias) v += *(const f32x4 *)(g.bias + col);
        if (EPI == EPI_RELU) {
          bf16x4 r;
#pragma unroll
          for (int i = 0; i < 4; ++i) r[i] = (bf16)fmaxf(v[i], 0.0f);
          *(bf16x4 *)(g.out_b + o) = r;
        } else if (EPI == EPI_RESID_RELU) {
          const bf16x4 h = *(const bf16x4 *)(g.resid + o);
          bf16x4 r, y;
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const float rl = fmaxf(v[i], 0.0f);
            r[i] = (bf16)rl;
            y[i] = (bf16)((float)h[i] + rl);
          }
          if (g.relu_out) *(bf16x4 *)(g.relu_out + o) = r;
          *(bf16x4 *)(g.out_b + o) = y;
        } else {
          *(f32x4 *)(g.out_f + o) = v;
          if (EPI == EPI_F32_MASK) {
            const bf16x4 m = *(const bf16x4 *)(g.mask + o);
            bf16x4 d;
#pragma unroll
            for (int i = 0; i < 4; ++i) d[i] = (bf16)((float)m[i] > 0.0f ? v[i] : 0.0f);
            *(bf16x4 *)(g.out_b + o) = d;
          }
        }
      }
    }
    t += (int)gridDim.x * W;
    if (t < tiles) gemm_rows<K, NE>(g, t, lr, lg, a);
  }
}

// ------------------------------------------------------- weight gradients
// Every matrix gradient A^T B (sums over the M rows) and bias gradient (column
// sums of B) of a backward pass in one launch: block (tile, split) forms one
// 64 x 64 tile of one matrix over its split's rows and writes a partial in the
// layout of the flat parameter vector; k_grad_reduce sums the splits in order
// (repeatable bits).  The matrices are small (54 tiles at four layers), so
// splitting the rows fills the chip: 28 us at 10 242 rows and four layers
// (one launch per matrix over 128 blocks took 23-33 us each, its own reduction
// and column sums 80 us more).
struct GradJob {
  const bf16 *A1, *A2;  // [M][K1], [M][K - K1] (null when K1 == K)
  const bf16 *B;        // [M][N]
  int K1, K, N;
  int tile0;            // first tile of the job
  long long off, boff;  // offsets of the matrix and its bias in the parameter vector
};
constexpr int GRAD_JOBS = 10;
struct GradArgs {
  GradJob job[GRAD_JOBS];
  int jobs, M, rows;    // rows of a split, a multiple of GRAD_CH
  long long n_params;
};
constexpr int GRAD_T = 64;    // tile edge
constexpr int GRAD_CH = 128;  // rows staged at a time

// 8x8 bf16 transpose: r[i] row i -> o[j] column j
__device__ __forceinline__ void transpose8(const uint4 (&r)[8], uint4 (&o)[8]) {
  const uint32_t *x = (const uint32_t *)r;
  uint32_t *y = (uint32_t *)o;
#pragma unroll
  for (int j = 0; j < 4; ++j)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const uint32_t lo = x[(2 * i) * 4 + j], hi = x[(2 * i + 1) * 4 + j];
      y[(2 * j) * 4 + i] = __builtin_amdgcn_perm(hi, lo, 0x05040100u);
      y[(2 * j + 1) * 4 + i] = __builtin_amdgcn_perm(hi, lo, 0x07060302u);
    }
}

__global__ void __launch_bounds__(256) k_grad(const GradArgs g, float *__restrict__ partial) {
  constexpr int LDM = GRAD_CH + 8;
  __shared__ __align__(16) bf16 s_t[2 * GRAD_T * LDM];  // A^T then B^T, [column][row]
  __shared__ float s_sum[GRAD_CH / 8][GRAD_T];
  int jn = 0;
#pragma unroll
  for (int i = 1; i < GRAD_JOBS; ++i)
    if (i < g.jobs && (int)blockIdx.x >= g.job[i].tile0) jn = i;
  const GradJob jb = g.job[jn];
  const int nt = jb.N / GRAD_T, tl = (int)blockIdx.x - jb.tile0;
  const int ti = tl / nt, tj = tl % nt;
  const int th = (int)threadIdx.x;
  // this thread's 8x8 block of the chunk: rows mb*8.., columns kb*8.. of A (threads 0..127) or B
  const bool isb = th >= 128;
  const int mb = th & 15, kb = (th >> 4) & 7;
  const bf16 *src;
  int ld;
  if (isb) {
    src = jb.B + tj * GRAD_T;
    ld = jb.N;
  } else if (ti * GRAD_T < jb.K1) {
    src = jb.A1 + ti * GRAD_T;
    ld = jb.K1;
  } else {
    src = jb.A2 + (ti * GRAD_T - jb.K1);
    ld = jb.K - jb.K1;
  }
  src += kb * 8;
  bf16 *dst = s_t + (isb ? GRAD_T * LDM : 0) + (kb * 8) * LDM + mb * 8;
  const int w = th >> 6, l = th & 63, lr = l & 15, lg = l >> 4;
  const int kt = (w >> 1) * 32, ct = (w & 1) * 32;  // this wavefront's 32 x 32 of the tile
  f32x4 acc[2][2];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  float sum[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
  const int m_lo = (int)blockIdx.y * g.rows, m_hi = min(g.M, m_lo + g.rows);
  uint4 r[8], o[8];
  auto load = [&](int m0) {
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const int m = m0 + mb * 8 + i;
      r[i] = m < m_hi ? *(const uint4 *)(src + (size_t)m * ld) : uint4{0u, 0u, 0u, 0u};
    }
  };
  load(m_lo);
  for (int m0 = m_lo; m0 < m_hi; m0 += GRAD_CH) {
    transpose8(r, o);
    if (ti == 0 && isb) {
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const bf16x8 col = __builtin_bit_cast(bf16x8, o[j]);
#pragma unroll
        for (int i = 0; i < 8; ++i) sum[j] += (float)col[i];
      }
    }
    __syncthreads();  // the chunk before this one has been read
#pragma unroll
    for (int j = 0; j < 8; ++j) *(uint4 *)(dst + j * LDM) = o[j];
    __syncthreads();
    if (m0 + GRAD_CH < m_hi) load(m0 + GRAD_CH);  // in flight under the products
#pragma unroll
    for (int q = 0; q < GRAD_CH / 32; ++q) {
      bf16x8 av[2], bv[2];
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        av[i] = *(const bf16x8 *)(s_t + (kt + i * 16 + lr) * LDM + q * 32 + lg * 8);
        bv[i] = *(const bf16x8 *)(s_t + (GRAD_T + ct + i * 16 + lr) * LDM + q * 32 + lg * 8);
      }
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) acc[i][j] = mfma(av[i], bv[j], acc[i][j]);
    }
  }
  float *out = partial + (size_t)blockIdx.y * g.n_params;
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int e = 0; e < 4; ++e)
        out[jb.off + (size_t)(ti * GRAD_T + kt + i * 16 + lg * 4 + e) * jb.N + tj * GRAD_T + ct + j * 16 + lr] =
            acc[i][j][e];
  if (ti == 0) {
    if (isb)
#pragma unroll
      for (int j = 0; j < 8; ++j) s_sum[mb][kb * 8 + j] = sum[j];
    __syncthreads();
    if (th < GRAD_T) {
      float s = 0.f;
#pragma unroll
      for (int i = 0; i < GRAD_CH / 8; ++i) s += s_sum[i][th];
      out[jb.boff + tj * GRAD_T + th] = s;
    }
  }
}

// grads[i] = sum over splits of partial[split][i], ascending
__global__ void __launch_bounds__(256) k_grad_reduce(const float *__restrict__ partial, int splits, int n,
                                                     float *__restrict__ out) {
  const int i = (int)(blockIdx.x * 256 + threadIdx.x);
  if (i >= n) return;
  float s = 0.0f;
  int b = 0;
  for (; b + 8 <= splits; b += 8) {
    float v[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) v[u] = partial[(size_t)(b + u) * n + i];
#pragma unroll
    for (int u = 0; u < 8; ++u) s += v[u];
  }
  for (; b < splits; ++b) s += partial[(size_t)b * n + i];
  out[i] = s;
}

// ---------------------------------------------------------- mesh kernels
// Lane k of wavefront (block*4 + w) owns row k of one cell or edge.
__device__ __forceinline__ int ent4() {
  return __builtin_amdgcn_readfirstlane(curve_block() * 4 + (int)(threadIdx.x >> 6));
}
__device__ __forceinline__ int lane() { return (int)(threadIdx.x & 63); }
// element k of row e of a dycore array (rows rs floats apart; lanes k >= rs
// read the row's last element, as the dycore kernels do)
__device__ __forceinline__ size_t rowi(int e, int k, int rs) { return (size_t)e * rs + (k < rs ? k : rs - 1); }
__device__ __forceinline__ float rowv(const float *p, int e, int k, int rs) { return p[rowi(e, k, rs)]; }

// Least-squares cell wind from the normal velocities of the cell's edges:
// minimise sum_s (n_s . U - u_s)^2, n_s = (cos a_s, sin a_s).
template <int NE>
__device__ __forceinline__ void lsq_frame(const Instance &I, int c, float &i11, float &i12, float &i22, int *eo,
                                          float *cs, float *sn, int &n) {
  n = I.m.neoc[c];
  float m11 = 0.f, m12 = 0.f, m22 = 0.f;
#pragma unroll
  for (int s = 0; s < NE; ++s) {
    eo[s] = I.m.eoc[c * NE + s];
    cs[s] = 0.f;
    sn[s] = 0.f;
    if (s < n) {
      cs[s] = I.m.cosang[eo[s]];
      sn[s] = I.m.sinang[eo[s]];
      m11 += cs[s] * cs[s];
      m12 += cs[s] * sn[s];
      m22 += sn[s] * sn[s];
    }
  }
  const float det = m11 * m22 - m12 * m12;
  i11 = m22 / det;
  i12 = -m12 / det;
  i22 = m11 / det;
}

// Feature columns of the published state (raw, before normalisation).
template <int NE>
__device__ __forceinline__ void raw_features(const Instance &I, int c, int k, float raw[6]) {
  const Work &B = I.b;
  const int n = I.m.neoc[c];
  int eo[NE];
#pragma unroll
  for (int s = 0; s < NE; ++s) eo[s] = I.m.eoc[c * NE + s];
  // every load first (slot tables are padded, so each slot is readable); the
  // least-squares frame and sums below are lsq_frame's, in the same order
  float u[NE], ca[NE], sa[NE], fe[NE];
#pragma unroll
  for (int s = 0; s < NE; ++s) {
    u[s] = rowv(B.p_u, eo[s], k, I.n.RS);
    ca[s] = I.m.cosang[eo[s]];
    sa[s] = I.m.sinang[eo[s]];
    fe[s] = I.m.fedge[eo[s]];
  }
  const float wk = rowv(B.p_w, c, k, I.n.RS), thk = rowv(B.p_theta, c, k, I.n.RS), rk = rowv(B.rho, c, k, I.n.RS);
  const float qk = I.n.NT > 0 ? rowv(B.q, c, k, I.n.RS) : 0.0f;
  float m11 = 0.f, m12 = 0.f, m22 = 0.f;
#pragma unroll
  for (int s = 0; s < NE; ++s)
    if (s < n) {
      m11 += ca[s] * ca[s];
      m12 += ca[s] * sa[s];
      m22 += sa[s] * sa[s];
    }
  const float det = m11 * m22 - m12 * m12;
  const float i11 = m22 / det, i12 = -m12 / det, i22 = m11 / det;
  float b1 = 0.f, b2 = 0.f, fs = 0.f;
#pragma unroll
  for (int s = 0; s < NE; ++s)
    if (s < n) {
      b1 += ca[s] * u[s];
      b2 += sa[s] * u[s];
      fs += fe[s];
    }
  const int L = I.n.L;
  raw[CH_UE] = (k < L) ? i11 * b1 + i12 * b2 : (k == L ? fs / (float)n : 0.0f);
  raw[CH_UN] = (k < L) ? i12 * b1 + i22 * b2 : 0.0f;
  raw[CH_W] = (k <= L) ? wk : 0.0f;
  raw[CH_TH] = (k < L) ? thk : 0.0f;
  raw[CH_RHO] = (k < L) ? rk : 0.0f;
  raw[CH_QV] = (k < L && I.n.NT > 0) ? qk : 0.0f;
}

template <int NE>
__global__ void __launch_bounds__(256) k_features(const Instance I, const float *__restrict__ mean,
                                                  const float *__restrict__ scale, bf16 *__restrict__ X,
                                                  float *__restrict__ raw_out) {
  const int c = ent4();
  if (c >= I.n.C) return;
  const int k = lane();
  float raw[6];
  raw_features<NE>(I, c, k, raw);
#pragma unroll
  for (int ch = 0; ch < 6; ++ch) {
    const int j = ch * HX_ROW + k;
    X[(size_t)c * KIN + j] = (bf16)((raw[ch] - mean[j]) * scale[j]);
    if (raw_out) raw_out[(size_t)c * KIN + j] = raw[ch];
  }
}

// dH_l = dH_{l+1} + dZ[:, :128] + sum over cellsOnCell j of dZ_j[128:] / n_j
// (the mean's adjoint; cellsOnCell is symmetric on a Voronoi mesh), and the
// next matrix gradient's operand dP = dH_l * [mask > 0] in bf16.  The encoder
// reads dP only (dH null).
template <int NE>
__global__ void __launch_bounds__(256) k_aggregate_back(const Instance I, const float *__restrict__ dHnext,
                                                        const float *__restrict__ dZ, const bf16 *__restrict__ mask,
                                                        float *__restrict__ dH, bf16 *__restrict__ dP) {
  const int c = ent4();
  if (c >= I.n.C) return;
  const int k = lane();
  const int n = I.m.neoc[c];
  float z0[NE], z1[NE], nj[NE];
#pragma unroll
  for (int s = 0; s < NE; ++s) {
    const int j = I.m.coc[c * NE + s];
    nj[s] = (float)I.m.neoc[j];
    z0[s] = dZ[(size_t)j * 2 * HID + HID + k];
    z1[s] = dZ[(size_t)j * 2 * HID + HID + 64 + k];
  }
  const size_t o = (size_t)c * HID;
  const float h0 = dHnext[o + k], h1 = dHnext[o + 64 + k];
  const float s0 = dZ[(size_t)c * 2 * HID + k], s1 = dZ[(size_t)c * 2 * HID + 64 + k];
  const float m0 = (float)mask[o + k], m1 = (float)mask[o + 64 + k];
  float a0 = 0.f, a1 = 0.f;
#pragma unroll
  for (int s = 0; s < NE; ++s)
    if (s < n) {
      const float inv = 1.0f / nj[s];
      a0 += z0[s] * inv;
      a1 += z1[s] * inv;
    }
  const float d0 = (h0 + s0) + a0, d1 = (h1 + s1) + a1;
  if (dH) {
    dH[o + k] = d0;
    dH[o + 64 + k] = d1;
  }
  dP[o + k] = (bf16)(m0 > 0.0f ? d0 : 0.0f);
  dP[o + 64 + k] = (bf16)(m1 > 0.0f ? d1 : 0.0f);
}

// Published fields of the coarse and fine handles that the target reads.
struct TargetArgs {
  int C, E, L, RS;
  const float *th_c, *rho_c, *w_c, *u_c;
  const float *th_f, *rho_f, *w_f, *u_f;
};

// normalised targets: (fine - coarse) / scale on the published states
__global__ void __launch_bounds__(256) k_target_cells(const TargetArgs a, const float *__restrict__ oscale,
                                                      float *__restrict__ Tc) {
  const int c = ent4();
  if (c >= a.C) return;
  const int k = lane();
  const int L = a.L;
  const float th = k < L ? (rowv(a.th_f, c, k, a.RS) - rowv(a.th_c, c, k, a.RS)) / oscale[O_TH * 64 + k] : 0.f;
  const float rh = k < L ? (rowv(a.rho_f, c, k, a.RS) - rowv(a.rho_c, c, k, a.RS)) / oscale[O_RHO * 64 + k] : 0.f;
  const float ww = (k >= 1 && k < L) ? (rowv(a.w_f, c, k, a.RS) - rowv(a.w_c, c, k, a.RS)) / oscale[O_W * 64 + k] : 0.f;
  float *t = Tc + (size_t)c * 3 * HX_ROW;
  t[k] = th;
  t[HX_ROW + k] = rh;
  t[2 * HX_ROW + k] = ww;
}

__global__ void __launch_bounds__(256) k_target_edges(const TargetArgs a, const float *__restrict__ oscale,
                                                      float *__restrict__ Te) {
  const int e = ent4();
  if (e >= a.E) return;
  const int k = lane();
  Te[(size_t)e * HX_ROW + k] = k < a.L ? (rowv(a.u_f, e, k, a.RS) - rowv(a.u_c, e, k, a.RS)) / oscale[O_UE * 64 + k] : 0.f;
}

__device__ __forceinline__ float wave_sum_f(float x) {
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) x += __shfl_down(x, off, 64);
  return x;
}

// normal-wind prediction of an edge from its two cells' outputs (normalised units)
__device__ __forceinline__ float edge_pred(const Instance &I, const float *Y, int e, int k) {
  const int c0 = I.m.coe[2 * e], c1 = I.m.coe[2 * e + 1];
  const float ue = 0.5f * (Y[(size_t)c0 * NOUT + O_UE * 64 + k] + Y[(size_t)c1 * NOUT + O_UE * 64 + k]);
  const float un = 0.5f * (Y[(size_t)c0 * NOUT + O_UN * 64 + k] + Y[(size_t)c1 * NOUT + O_UN * 64 + k]);
  return I.m.cosang[e] * ue + I.m.sinang[e] * un;
}

// g_e = dLoss/d(du_e) and the per-block partial sum of squared errors
__global__ void __launch_bounds__(256) k_loss_edges(const Instance I, const float *__restrict__ Y,
                                                    const float *__restrict__ Te, float *__restrict__ g,
                                                    float *__restrict__ lpart, float inv_n) {
  __shared__ float s_part[4];
  const int e = ent4();
  const int k = lane();
  float d2 = 0.f;
  if (e < I.n.E) {
    float gv = 0.f;
    if (k < I.n.L) {
      const float d = edge_pred(I, Y, e, k) - Te[(size_t)e * HX_ROW + k];
      gv = 2.0f * d * inv_n;
      d2 = d * d;
    }
    g[(size_t)e * HX_ROW + k] = gv;
  }
  d2 = wave_sum_f(d2);
  if (k == 0) s_part[threadIdx.x >> 6] = d2;
  __syncthreads();
  if (threadIdx.x == 0) lpart[curve_block()] = ((s_part[0] + s_part[1]) + s_part[2]) + s_part[3];
}

// dY of every output channel (bf16) and the per-block partial sums of squared
// errors of theta, rho and w; the wind channels gather the edge gradients
template <int NE>
__global__ void __launch_bounds__(256) k_loss_cells(const Instance I, const float *__restrict__ Y,
                                                    const float *__restrict__ Tc, const float *__restrict__ g,
                                                    bf16 *__restrict__ dY, float *__restrict__ lpart,
                                                    float inv_nc, float inv_nw) {
  __shared__ float s_part[3][4];
  const int c = ent4();
  const int k = lane();
  const int L = I.n.L;
  float d2[3] = {0.f, 0.f, 0.f};
  if (c < I.n.C) {
    const float *y = Y + (size_t)c * NOUT;
    const float *t = Tc + (size_t)c * 3 * HX_ROW;
    bf16 *dy = dY + (size_t)c * NOUT;
    const int n = I.m.neoc[c];
    float ge = 0.f, gn = 0.f;
#pragma unroll
    for (int s = 0; s < NE; ++s) {
      if (s < n) {
        const int e = I.m.eoc[c * NE + s];
        const float gv = 0.5f * g[(size_t)e * HX_ROW + k];
        ge += I.m.cosang[e] * gv;
        gn += I.m.sinang[e] * gv;
      }
    }
    dy[O_UE * 64 + k] = (bf16)(k < L ? ge : 0.f);
    dy[O_UN * 64 + k] = (bf16)(k < L ? gn : 0.f);
    const bool lay = k < L, intr = k >= 1 && k < L;
    const float dth = lay ? y[O_TH * 64 + k] - t[k] : 0.f;
    const float drh = lay ? y[O_RHO * 64 + k] - t[HX_ROW + k] : 0.f;
    const float dw = intr ? y[O_W * 64 + k] - t[2 * HX_ROW + k] : 0.f;
    dy[O_TH * 64 + k] = (bf16)(2.0f * dth * inv_nc);
    dy[O_RHO * 64 + k] = (bf16)(2.0f * drh * inv_nc);
    dy[O_W * 64 + k] = (bf16)(2.0f * dw * inv_nw);
    d2[0] = dth * dth;
    d2[1] = drh * drh;
    d2[2] = dw * dw;
  }
#pragma unroll
  for (int v = 0; v < 3; ++v) {
    const float x = wave_sum_f(d2[v]);
    if (k == 0) s_part[v][threadIdx.x >> 6] = x;
  }
  __syncthreads();
  if (threadIdx.x < 3) {
    const int v = (int)threadIdx.x;
    lpart[(size_t)v * gridDim.x + curve_block()] = ((s_part[v][0] + s_part[v][1]) + s_part[v][2]) + s_part[v][3];
  }
}

// The four loss sums (edges, then theta, rho and w of the cells) in binary64,
// one block each: a thread's strided partials, then a fixed tree.
__global__ void __launch_bounds__(1024) k_loss_sums(const float *__restrict__ p, int ne, int nc,
                                                    double *__restrict__ out) {
  __shared__ double s_sum[1024];
  const int v = (int)blockIdx.x, t = (int)threadIdx.x;
  const int n = v == 0 ? ne : nc;
  if (v > 0) p += (size_t)ne + (size_t)(v - 1) * nc;
  double s = 0.0;
#pragma unroll 4
  for (int b = t; b < n; b += 1024) s += (double)p[b];
  s_sum[t] = s;
  __syncthreads();
  for (int off = 512; off >= 1; off >>= 1) {
    if (t < off) s_sum[t] = s_sum[t] + s_sum[t + off];
    __syncthreads();
  }
  if (t == 0) out[v] = s_sum[0];
}

// ---------------------------------------------------------- application
// Per-block partials of sum_c,k area * dzw * drho (the raw density
// correction) and of the volume sum_c,k area * dzw.
__global__ void __launch_bounds__(256) k_mass_partial(const Instance I, const float *__restrict__ Y,
                                                      const float *__restrict__ oscale, double *__restrict__ part) {
  __shared__ double s_part[2][4];
  const int c = ent4();
  const int k = lane();
  double v = 0.0, vol = 0.0;
  if (c < I.n.C && k < I.n.L) {
    const double dr = (double)(Y[(size_t)c * NOUT + O_RHO * 64 + k] * oscale[O_RHO * 64 + k]);
    vol = (1.0 / (double)I.m.invarea[c]) * (1.0 / (double)I.z.rdzw[k]);
    v = vol * dr;
  }
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) {
    v += __shfl_down(v, off, 64);
    vol += __shfl_down(vol, off, 64);
  }
  if (k == 0) {
    s_part[0][threadIdx.x >> 6] = v;
    s_part[1][threadIdx.x >> 6] = vol;
  }
  __syncthreads();
  if (threadIdx.x < 2)
    part[(size_t)threadIdx.x * gridDim.x + curve_block()] =
        ((s_part[threadIdx.x][0] + s_part[threadIdx.x][1]) + s_part[threadIdx.x][2]) + s_part[threadIdx.x][3];
}

// shift = (sum of the correction partials) / (sum of the volume partials),
// one block, fixed order
__global__ void __launch_bounds__(256) k_mass_shift(const double *__restrict__ part, int nb,
                                                    float *__restrict__ shift) {
  __shared__ double s[2][256];
  const int t = (int)threadIdx.x;
  double a = 0.0, b = 0.0;
  for (int i = t; i < nb; i += 256) {
    a += part[i];
    b += part[(size_t)nb + i];
  }
  s[0][t] = a;
  s[1][t] = b;
  __syncthreads();
  for (int off = 128; off >= 1; off >>= 1) {
    if (t < off) {
      s[0][t] = s[0][t] + s[0][t + off];
      s[1][t] = s[1][t] + s[1][t + off];
    }
    __syncthreads();
  }
  if (t == 0) shift[0] = (float)(s[0][0] / s[1][0]);
}

// cells: rho' = rho + drho - shift, theta' = theta + dtheta, rtheta' = rho' theta',
// rw' = rw + dw * (fzm rho'_k + fzp rho'_{k-1}) (fzm zz_k + fzp zz_{k-1}) inside the column
__global__ void __launch_bounds__(256) k_apply_cells(const Instance I, const float *__restrict__ Y,
                                                     const float *__restrict__ oscale, const float *__restrict__ shift,
                                                     float gain) {
  const int c = ent4();
  if (c >= I.n.C) return;
  const int k = lane();
  const int L = I.n.L;
  const Work &B = I.b;
  const float *y = Y + (size_t)c * NOUT;
  const size_t o = rowi(c, k, I.n.RS);
  float rho = B.rho[o];
  if (k < L) {
    const float drho = gain * (y[O_RHO * 64 + k] * oscale[O_RHO * 64 + k] - shift[0]);
    const float th = B.p_theta[o] + gain * (y[O_TH * 64 + k] * oscale[O_TH * 64 + k]);
    rho = rho + drho;
    B.rho[o] = rho;
    B.rt[o] = rho * th;
  }
  const float rho_m = __shfl_up(rho, 1, 64);
  const float zk = I.z.zz[o];
  const float zkm = __shfl_up(zk, 1, 64);
  if (k >= 1 && k < L) {
    const float fzm = I.z.fzm[k], fzp = I.z.fzp[k];
    const float dw = gain * (y[O_W * 64 + k] * oscale[O_W * 64 + k]);
    B.rw[o] = B.rw[o] + dw * ((fzm * rho + fzp * rho_m) * (fzm * zk + fzp * zkm));
  }
}

// edges (after the cells): u' = u + du, ru' = (rho'_0 + rho'_1)/2 u', and
// the carried u recomputed from ru' as the diagnostic rebuild forms it,
// 2 ru' / (rho'_0 + rho'_1)
__global__ void __launch_bounds__(256) k_apply_edges(const Instance I, const float *__restrict__ Y,
                                                     const float *__restrict__ oscale, float gain) {
  const int e = ent4();
  if (e >= I.n.E) return;
  const int k = lane();
  if (k >= I.n.L) return;
  const int c0 = I.m.coe[2 * e], c1 = I.m.coe[2 * e + 1];
  const size_t o = rowi(e, k, I.n.RS);
  const float u = I.b.p_u[o] + gain * (edge_pred(I, Y, e, k) * oscale[O_UE * 64 + k]);
  const float r0 = rowv(I.b.rho, c0, k, I.n.RS), r1 = rowv(I.b.rho, c1, k, I.n.RS);
  const float ru = (0.5f * (r0 + r1)) * u;
  I.b.ru[o] = ru;
  I.b.p_u[o] = (2.0f * ru) / (r0 + r1);
}

// ---------------------------------------------------------- checks
__device__ __forceinline__ float nanmax(float a, float b) { return (b != b || b > a) ? b : a; }

// Per-block partials of the checks: max |u| dt / dc (horizontal CFL),
// max |w| dt rdzw / zz (vertical CFL), max |divergence| dt (a NaN anywhere
// wins), and the dry mass sum areaCell * dzw * rho_zz in binary64.
template <int NE>
__global__ void __launch_bounds__(256) k_checks_cells(const Instance I, float dt, float *__restrict__ fpart,
                                                      double *__restrict__ mpart) {
  __shared__ float s_f[3][4];
  __shared__ double s_m[4];
  const int c = ent4();
  const int k = lane();
  const int L = I.n.L;
  const Work &B = I.b;
  float div = 0.f, cfl = 0.f, vc = 0.f;
  double mass = 0.0;
  if (c < I.n.C) {
    const int n = I.m.neoc[c];
    // every load first (slot tables are padded, so each slot is readable),
    // then the sums in slot order
    int e[NE];
#pragma unroll
    for (int s = 0; s < NE; ++s) e[s] = I.m.eoc[c * NE + s];
    float u[NE], sd[NE], idc[NE];
#pragma unroll
    for (int s = 0; s < NE; ++s) {
      u[s] = rowv(B.p_u, e[s], k, I.n.RS);
      sd[s] = I.m.csdv[c * NE + s];
      idc[s] = I.m.invdc[e[s]];
    }
    const float wk = rowv(B.p_w, c, k, I.n.RS), zk = rowv(I.z.zz, c, k, I.n.RS), rk = rowv(B.rho, c, k, I.n.RS);
    const float rdzw = I.z.rdzw[k];
#pragma unroll
    for (int s = 0; s < NE; ++s) {
      if (s < n) {
        div += sd[s] * u[s];
        cfl = nanmax(cfl, fabsf(u[s]) * dt * idc[s]);
      }
    }
    div = fabsf(div * I.m.invarea[c]) * dt;
    if (k >= 1 && k < L) vc = fabsf(wk) * dt * rdzw / zk;
    if (k < L) mass = (1.0 / (double)I.m.invarea[c]) * (1.0 / (double)rdzw) * (double)rk;
    if (k >= L) {
      div = 0.f;
      cfl = 0.f;
    }
  }
  for (int off = 32; off >= 1; off >>= 1) {
    cfl = nanmax(cfl, __shfl_down(cfl, off, 64));
    vc = nanmax(vc, __shfl_down(vc, off, 64));
    div = nanmax(div, __shfl_down(div, off, 64));
    mass += __shfl_down(mass, off, 64);
  }
  const int w = (int)(threadIdx.x >> 6);
  if (k == 0) {
    s_f[0][w] = cfl;
    s_f[1][w] = vc;
    s_f[2][w] = div;
    s_m[w] = mass;
  }
  __syncthreads();
  if (threadIdx.x < 3) {
    const int v = (int)threadIdx.x;
    fpart[(size_t)v * gridDim.x + curve_block()] = nanmax(nanmax(nanmax(s_f[v][0], s_f[v][1]), s_f[v][2]), s_f[v][3]);
  } else if (threadIdx.x == 3) {
    mpart[curve_block()] = ((s_m[0] + s_m[1]) + s_m[2]) + s_m[3];
  }
}

// one block: out = {cfl_h, cfl_v, div (floats), dry mass (double)} from the
// partials in a fixed order
__global__ void __launch_bounds__(256) k_checks_final(const float *__restrict__ fpart, const double *__restrict__ mpart,
                                                      int nb, float *__restrict__ fout, double *__restrict__ mout) {
  __shared__ float s_f[3][256];
  __shared__ double s_m[256];
  const int t = (int)threadIdx.x;
  float f[3] = {0.f, 0.f, 0.f};
  double m = 0.0;
  for (int b = t; b < nb; b += 256) {
#pragma unroll
    for (int v = 0; v < 3; ++v) f[v] = nanmax(f[v], fpart[(size_t)v * nb + b]);
    m += mpart[b];
  }
#pragma unroll
  for (int v = 0; v < 3; ++v) s_f[v][t] = f[v];
  s_m[t] = m;
  __syncthreads();
  for (int off = 128; off >= 1; off >>= 1) {
    if (t < off) {
#pragma unroll
      for (int v = 0; v < 3; ++v) s_f[v][t] = nanmax(s_f[v][t], s_f[v][t + off]);
      s_m[t] = s_m[t] + s_m[t + off];
    }
    __syncthreads();
  }
  if (t == 0) {
#pragma unroll
    for (int v = 0; v < 3; ++v) fout[v] = s_f[v][0];
    mout[0] = s_m[0];
  }
}

// ---------------------------------------------------------- optimiser
struct Seg {
  long long off;   // offset in the flat fp32 parameter vector
  int K, N;        // matrix shape (N = count, K = 1 for a bias)
  long long boff;  // offset in the bf16 weight buffers (matrices only, -1 for biases)
};
constexpr int MAX_SEGS = 2 * (8 + 2);
struct SegTable {
  Seg seg[MAX_SEGS];
  int n;
};

// bf16 copies of parameter i where it belongs to a matrix: W[k][n] (backward)
// and Wt[n][k] (forward).  A block of 256 parameters lies in one segment, or
// in few: the table is walked with uniform reads.
__device__ __forceinline__ void store_weight(const SegTable &t, long long i, float p, bf16 *__restrict__ W,
                                             bf16 *__restrict__ Wt) {
  for (int s = 0; s < t.n; ++s) {
    const Seg sg = t.seg[s];
    const long long j = i - sg.off;
    if (sg.boff < 0 || j < 0 || j >= (long long)sg.K * sg.N) continue;
    const int k = (int)j / sg.N, n = (int)j % sg.N;
    const bf16 b = (bf16)p;
    W[sg.boff + j] = b;
    Wt[sg.boff + (long long)n * sg.K + k] = b;
  }
}

__global__ void __launch_bounds__(256) k_adam(float *__restrict__ p, const float *__restrict__ g,
                                              float *__restrict__ m, float *__restrict__ v, size_t n, float lr,
                                              float b1, float b2, float eps, float bc1, float bc2, const SegTable t,
                                              bf16 *__restrict__ W, bf16 *__restrict__ Wt) {
  const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= n) return;
  const float gi = g[i];
  const float mi = b1 * m[i] + (1.0f - b1) * gi;
  const float vi = b2 * v[i] + (1.0f - b2) * (gi * gi);
  m[i] = mi;
  v[i] = vi;
  const float mh = mi / bc1, vh = vi / bc2;
  const float pn = p[i] - lr * (mh / (sqrtf(vh) + eps));
  p[i] = pn;
  store_weight(t, (long long)i, pn, W, Wt);
}

// bf16 copies of every weight matrix
__global__ void __launch_bounds__(256) k_weights(const float *__restrict__ p, size_t n, const SegTable t,
                                                 bf16 *__restrict__ W, bf16 *__restrict__ Wt) {
  const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
  if (i < n) store_weight(t, (long long)i, p[i], W, Wt);
}

// logical (original) order export of per-cell rows of width w
__global__ void __launch_bounds__(256) k_export_rows(const float *__restrict__ src, const int *__restrict__ old_of_new,
                                                     int n, int w, float *__restrict__ dst) {
  const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= (size_t)n * w) return;
  const int r = (int)(i / w), j = (int)(i % w);
  dst[(size_t)old_of_new[r] * w + j] = src[i];
}

__global__ void __launch_bounds__(256) k_export_rows_bf16(const bf16 *__restrict__ src,
                                                          const int *__restrict__ old_of_new, int n, int w,
                                                          float *__restrict__ dst) {
  const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= (size_t)n * w) return;
  const int r = (int)(i / w), j = (int)(i % w);
  dst[(size_t)old_of_new[r] * w + j] = (float)src[i];
}

inline unsigned nblk(size_t n, int per = 256) { return (unsigned)((n + per - 1) / per); }

}  // namespace

// ====================================================================== Net
struct Net {
  int C = 0, E = 0, NL = 0, NE = 6;
  int cus = 256;
  SegTable table{};
  int splits = 1, split_rows = 128;  // of the weight gradients
  std::vector<void *> allocs;
  std::vector<Seg> segs;  // W_in, b_in, (W_l, b_l) x NL, W_out, b_out
  size_t n_params = 0, n_bf = 0;
  float *params = nullptr, *grads = nullptr, *adam_m = nullptr, *adam_v = nullptr;
  bf16 *w_bf = nullptr, *wt_bf = nullptr;
  float *in_mean = nullptr, *in_scale = nullptr, *out_scale = nullptr;
  bf16 *X = nullptr;
  std::vector<bf16 *> H, A, R;  // H: NL+1, A and R: NL
  float *Y = nullptr;
  float *Tc = nullptr, *Te = nullptr, *g = nullptr;
  bf16 *dY = nullptr;
  std::vector<bf16 *> dP;       // masked gradients: encoder, then the layers
  float *dH0 = nullptr, *dH1 = nullptr, *dZ = nullptr;
  float *partial = nullptr, *lpart = nullptr;
  double *loss_out = nullptr, *mpart = nullptr;
  float *shift = nullptr, *checks = nullptr, *raw = nullptr, *cpart = nullptr;
  double *mass_out = nullptr;
  float check_host[6];  // three maxima, pad, then the binary64 mass
  int have_target = 0, have_forward = 0;
  std::string error;

  template <class T> int alloc(T **p, size_t count) {
    void *q = nullptr;
    if (hipMalloc(&q, std::max<size_t>(count, 1) * sizeof(T)) != hipSuccess) return -1;
    if (hipMemset(q, 0, std::max<size_t>(count, 1) * sizeof(T)) != hipSuccess) return -1;
    allocs.push_back(q);
    *p = (T *)q;
    return 0;
  }
  ~Net() {
    for (void *p : allocs) (void)hipFree(p);
  }
  const Seg &w_in() const { return segs[0]; }
  const Seg &b_in() const { return segs[1]; }
  const Seg &w_l(int l) const { return segs[2 + 2 * l]; }
  const Seg &b_l(int l) const { return segs[3 + 2 * l]; }
  const Seg &w_out() const { return segs[2 + 2 * NL]; }
  const Seg &b_out() const { return segs[3 + 2 * NL]; }
  const bf16 *Wt(const Seg &s) const { return wt_bf + s.boff; }
  const bf16 *W(const Seg &s) const { return w_bf + s.boff; }
  const float *P(const Seg &s) const { return params + s.off; }
  float *G(const Seg &s) const { return grads + s.off; }
};

namespace {

template <class KFn>
int set_lds(KFn fn, size_t bytes) {
  return hipFuncSetAttribute((const void *)fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes) ==
                 hipSuccess
             ? 0
             : -1;
}

// Wavefronts per block: 4, so that a few thousand rows still reach every CU;
// 8 (two blocks of them per CU share its LDS) once every CU has a block of 8.
template <int K, int N, int NC, int EPI, int NE>
int gemm(const Net &n, const GemmArgs &g, hipStream_t s) {
  const size_t lds = (size_t)NC * (K + 8) * sizeof(bf16);
  static const int ready = set_lds(k_gemm<K, N, NC, EPI, NE>, lds);
  if (ready) return -1;
  const int tiles = (g.M + 15) / 16;
  const int W = tiles >= 8 * n.cus ? 8 : 4;
  const int per_cu = std::max(1, (int)((size_t)160 * 1024 / lds));
  const int grid = std::max(1, std::min((tiles + W - 1) / W, n.cus * std::min(per_cu, 4)));
  if (g_prof_on) prof_mark("k_net_gemm", s, 1);
  hipLaunchKernelGGL((k_gemm<K, N, NC, EPI, NE>), dim3(grid, N / NC), dim3(64 * W), lds, s, g);
  if (g_prof_on) prof_mark("k_net_gemm", s, 0);
  return hipGetLastError() == hipSuccess ? 0 : -1;
}

#define NE_LAUNCH(NEV, KERN, grid, block, s, ...)                                   \
  do {                                                                              \
    if ((NEV) == 6)                                                                 \
      hipLaunchKernelGGL(KERN<6>, dim3(grid), dim3(block), 0, s, __VA_ARGS__);      \
    else                                                                            \
      hipLaunchKernelGGL(KERN<7>, dim3(grid), dim3(block), 0, s, __VA_ARGS__);      \
  } while (0)

}  // namespace

int features(Net &n, const Instance &I, hipStream_t s, float *raw = nullptr) {
  if (g_prof_on) prof_mark("k_net_features", s, 1);
  NE_LAUNCH(n.NE, k_features, nblk(n.C, 4), 256, s, I, (const float *)n.in_mean, (const float *)n.in_scale, n.X,
            raw);
  if (g_prof_on) prof_mark("k_net_features", s, 0);
  return hipGetLastError() == hipSuccess ? 0 : -1;
}

int forward(Net &n, const Instance &I, bool keep, hipStream_t s) {
  if (features(n, I, s)) return -1;
  GemmArgs g{};
  g.M = n.C;
  g.coc = I.m.coc;
  g.neoc = I.m.neoc;
  g.A = n.X;
  g.Bt = n.Wt(n.w_in());
  g.bias = n.P(n.b_in());
  g.out_b = n.H[0];
  if (gemm<KIN, HID, HID, EPI_RELU, 0>(n, g, s)) return -1;
  for (int l = 0; l < n.NL; ++l) {
    g.A = g.resid = n.H[l];
    g.Bt = n.Wt(n.w_l(l));
    g.bias = n.P(n.b_l(l));
    g.out_b = n.H[l + 1];
    g.relu_out = keep ? n.R[l] : nullptr;
    g.mean_out = keep ? n.A[l] : nullptr;
    if (n.NE == 6 ? gemm<2 * HID, HID, HID, EPI_RESID_RELU, 6>(n, g, s)
                  : gemm<2 * HID, HID, HID, EPI_RESID_RELU, 7>(n, g, s))
      return -1;
  }
  g = GemmArgs{};
  g.M = n.C;
  g.A = n.H[n.NL];
  g.Bt = n.Wt(n.w_out());
  g.bias = n.P(n.b_out());
  g.out_f = n.Y;
  if (gemm<HID, NOUT, NOUT / 4, EPI_F32, 0>(n, g, s)) return -1;
  n.have_forward = 1;
  return 0;
}

int loss(Net &n, const Instance &I, double *out4, hipStream_t s) {
  const int L = I.n.L;
  const unsigned ge = nblk(n.E, 4), gc = nblk(n.C, 4);
  hipLaunchKernelGGL(k_loss_edges, dim3(ge), dim3(256), 0, s, I, (const float *)n.Y, (const float *)n.Te, n.g,
                     n.lpart, 1.0f / (float)((double)n.E * L));
  NE_LAUNCH(n.NE, k_loss_cells, gc, 256, s, I, (const float *)n.Y, (const float *)n.Tc, (const float *)n.g, n.dY,
            n.lpart + ge, 1.0f / (float)((double)n.C * L), 1.0f / (float)((double)n.C * (L - 1)));
  hipLaunchKernelGGL(k_loss_sums, dim3(4), dim3(1024), 0, s, (const float *)n.lpart, (int)ge, (int)gc, n.loss_out);
  if (hipGetLastError() != hipSuccess) return -1;
  double raw[4];
  if (hipMemcpyAsync(raw, n.loss_out, sizeof raw, hipMemcpyDeviceToHost, s) != hipSuccess ||
      hipStreamSynchronize(s) != hipSuccess)
    return -1;
  out4[1] = raw[0] / ((double)n.E * L);
  out4[2] = raw[1] / ((double)n.C * L);
  out4[3] = raw[2] / ((double)n.C * L);
  out4[4] = raw[3] / ((double)n.C * (L - 1));
  out4[0] = ((out4[1] + out4[2]) + out4[3]) + out4[4];
  return 0;
}

// The gradient chain first (each pass leaves the masked bf16 gradient that its
// matrix needs), then every matrix and bias gradient in one launch.
int backward(Net &n, const Instance &I, hipStream_t s) {
  const int C = n.C, NL = n.NL;
  GemmArgs g{};
  g.M = C;
  g.A = n.dY;
  g.Bt = n.W(n.w_out());
  g.out_f = n.dH1;
  g.mask = n.R[NL - 1];
  g.out_b = n.dP[NL];
  if (gemm<NOUT, HID, HID, EPI_F32_MASK, 0>(n, g, s)) return -1;
  float *dHnext = n.dH1, *dHcur = n.dH0;
  for (int l = NL - 1; l >= 0; --l) {
    g = GemmArgs{};
    g.M = C;
    g.A = n.dP[l + 1];
    g.Bt = n.W(n.w_l(l));
    g.out_f = n.dZ;
    if (gemm<HID, 2 * HID, HID, EPI_F32, 0>(n, g, s)) return -1;
    NE_LAUNCH(n.NE, k_aggregate_back, nblk(C, 4), 256, s, I, (const float *)dHnext, (const float *)n.dZ,
              (const bf16 *)(l > 0 ? n.R[l - 1] : n.H[0]), l > 0 ? dHcur : nullptr, n.dP[l]);
    std::swap(dHnext, dHcur);
  }
  GradArgs a{};
  a.M = C;
  a.rows = n.split_rows;
  a.n_params = (long long)n.n_params;
  int tiles = 0;
  auto job = [&](const bf16 *A1, int K1, const bf16 *A2, const Seg &w, const Seg &b, const bf16 *B) {
    a.job[a.jobs++] = GradJob{A1, A2, B, K1, w.K, w.N, tiles, w.off, b.off};
    tiles += (w.K / GRAD_T) * (w.N / GRAD_T);
  };
  job(n.X, KIN, nullptr, n.w_in(), n.b_in(), n.dP[0]);
  for (int l = 0; l < NL; ++l) job(n.H[l], HID, n.A[l], n.w_l(l), n.b_l(l), n.dP[l + 1]);
  job(n.H[NL], HID, nullptr, n.w_out(), n.b_out(), n.dY);
  if (g_prof_on) prof_mark("k_net_grad", s, 1);
  hipLaunchKernelGGL(k_grad, dim3(tiles, n.splits), dim3(256), 0, s, a, n.partial);
  if (g_prof_on) prof_mark("k_net_grad", s, 0);
  hipLaunchKernelGGL(k_grad_reduce, dim3(nblk(n.n_params)), dim3(256), 0, s, (const float *)n.partial, n.splits,
                     (int)n.n_params, n.grads);
  return hipGetLastError() == hipSuccess ? 0 : -1;
}

int sync_bf16(Net &n, hipStream_t s) {
  hipLaunchKernelGGL(k_weights, dim3(nblk(n.n_params)), dim3(256), 0, s, (const float *)n.params, n.n_params, n.table,
                     n.w_bf, n.wt_bf);
  return hipGetLastError() == hipSuccess ? 0 : -1;
}

int adam(Net &n, float lr, float b1, float b2, float eps, int t, hipStream_t s) {
  const float bc1 = (float)(1.0 - std::pow((double)b1, t)), bc2 = (float)(1.0 - std::pow((double)b2, t));
  hipLaunchKernelGGL(k_adam, dim3(nblk(n.n_params)), dim3(256), 0, s, n.params, (const float *)n.grads, n.adam_m,
                     n.adam_v, n.n_params, lr, b1, b2, eps, bc1, bc2, n.table, n.w_bf, n.wt_bf);
  return hipGetLastError() == hipSuccess ? 0 : -1;
}

int target(Net &n, const Instance &Ic, const Instance &If, hipStream_t s) {
  const TargetArgs a{n.C, n.E, Ic.n.L, Ic.n.RS, Ic.b.p_theta, Ic.b.rho, Ic.b.p_w, Ic.b.p_u,
                     If.b.p_theta, If.b.rho, If.b.p_w, If.b.p_u};
  hipLaunchKernelGGL(k_target_cells, dim3(nblk(n.C, 4)), dim3(256), 0, s, a, (const float *)n.out_scale, n.Tc);
  hipLaunchKernelGGL(k_target_edges, dim3(nblk(n.E, 4)), dim3(256), 0, s, a, (const float *)n.out_scale, n.Te);
  n.have_target = 1;
  return hipGetLastError() == hipSuccess ? 0 : -1;
}

int apply(Net &n, const Instance &I, float gain, hipStream_t s) {
  const unsigned gc = nblk(n.C, 4);
  if (g_prof_on) prof_mark("k_net_apply", s, 1);
  hipLaunchKernelGGL(k_mass_partial, dim3(gc), dim3(256), 0, s, I, (const float *)n.Y, (const float *)n.out_scale,
                     n.mpart);
  hipLaunchKernelGGL(k_mass_shift, dim3(1), dim3(256), 0, s, (const double *)n.mpart, (int)gc, n.shift);
  hipLaunchKernelGGL(k_apply_cells, dim3(gc), dim3(256), 0, s, I, (const float *)n.Y, (const float *)n.out_scale,
                     (const float *)n.shift, gain);
  hipLaunchKernelGGL(k_apply_edges, dim3(nblk(n.E, 4)), dim3(256), 0, s, I, (const float *)n.Y,
                     (const float *)n.out_scale, gain);
  if (g_prof_on) prof_mark("k_net_apply", s, 0);
  return hipGetLastError() == hipSuccess ? 0 : -1;
}

int checks(Net &n, const Instance &I, float dt, float out[3], double *mass, hipStream_t s) {
  const unsigned gc = nblk(n.C, 4);
  if (g_prof_on) prof_mark("k_net_checks", s, 1);
  NE_LAUNCH(n.NE, k_checks_cells, gc, 256, s, I, dt, n.cpart, n.mpart);
  hipLaunchKernelGGL(k_checks_final, dim3(1), dim3(256), 0, s, (const float *)n.cpart, (const double *)n.mpart,
                     (int)gc, n.checks, n.mass_out);
  if (g_prof_on) prof_mark("k_net_checks", s, 0);
  if (hipGetLastError() != hipSuccess) return -1;
  // one host read: the three maxima and the binary64 mass side by side
  if (hipMemcpyAsync(n.check_host, n.checks, 4 * sizeof(float), hipMemcpyDeviceToHost, s) != hipSuccess ||
      hipMemcpyAsync(&n.check_host[4], n.mass_out, sizeof(double), hipMemcpyDeviceToHost, s) != hipSuccess ||
      hipStreamSynchronize(s) != hipSuccess)
    return -1;
  for (int v = 0; v < 3; ++v) out[v] = n.check_host[v];
  std::memcpy(mass, &n.check_host[4], sizeof(double));
  return 0;
}

Net *create(const Instance &I, int layers, std::string *err) {
  Net *n = new Net();
  n->C = I.n.C;
  n->E = I.n.E;
  n->NL = layers;
  n->NE = I.n.ME;
  int dev = 0, cus = 256;
  if (hipGetDevice(&dev) == hipSuccess) {
    hipDeviceProp_t prop;
    if (hipGetDeviceProperties(&prop, dev) == hipSuccess && prop.multiProcessorCount > 0)
      cus = prop.multiProcessorCount;
  }
  n->cus = cus;
  // parameter segments
  size_t off = 0, boff = 0;
  auto mat = [&](int K, int N) {
    n->segs.push_back({(long long)off, K, N, (long long)boff});
    off += (size_t)K * N;
    boff += (size_t)K * N;
  };
  auto vec = [&](int N) {
    n->segs.push_back({(long long)off, 1, N, -1});
    off += (size_t)N;
  };
  mat(KIN, HID);
  vec(HID);
  for (int l = 0; l < layers; ++l) {
    mat(2 * HID, HID);
    vec(HID);
  }
  mat(HID, NOUT);
  vec(NOUT);
  n->n_params = off;
  n->n_bf = boff;
  n->table.n = (int)n->segs.size();
  for (int i = 0; i < n->table.n; ++i) n->table.seg[i] = n->segs[i];
  // splits of the weight gradients: about 640 rows each, at most 32 (the
  // partials of a split are one parameter vector, 0.9 MB at four layers)
  n->splits = std::min(32, std::max(1, (n->C + 639) / 640));
  n->split_rows = ((n->C + n->splits - 1) / n->splits + GRAD_CH - 1) / GRAD_CH * GRAD_CH;
  n->splits = (n->C + n->split_rows - 1) / n->split_rows;
  const size_t C = (size_t)n->C, E = (size_t)n->E;
  int rc = 0;
  rc |= n->alloc(&n->params, off);
  rc |= n->alloc(&n->grads, off);
  rc |= n->alloc(&n->adam_m, off);
  rc |= n->alloc(&n->adam_v, off);
  rc |= n->alloc(&n->w_bf, boff);
  rc |= n->alloc(&n->wt_bf, boff);
  rc |= n->alloc(&n->in_mean, KIN);
  rc |= n->alloc(&n->in_scale, KIN);
  rc |= n->alloc(&n->out_scale, NOUT);
  rc |= n->alloc(&n->X, C * KIN);
  n->H.assign(layers + 1, nullptr);
  n->A.assign(layers, nullptr);
  n->R.assign(layers, nullptr);
  for (auto &p : n->H) rc |= n->alloc(&p, C * HID);
  for (auto &p : n->A) rc |= n->alloc(&p, C * HID);
  for (auto &p : n->R) rc |= n->alloc(&p, C * HID);
  rc |= n->alloc(&n->Y, C * NOUT);
  rc |= n->alloc(&n->Tc, C * 3 * HX_ROW);
  rc |= n->alloc(&n->Te, E * HX_ROW);
  rc |= n->alloc(&n->g, E * HX_ROW);
  rc |= n->alloc(&n->dY, C * NOUT);
  n->dP.assign(layers + 1, nullptr);
  for (auto &p : n->dP) rc |= n->alloc(&p, C * HID);
  rc |= n->alloc(&n->dH0, C * HID);
  rc |= n->alloc(&n->dH1, C * HID);
  rc |= n->alloc(&n->dZ, C * 2 * HID);
  rc |= n->alloc(&n->partial, (size_t)n->splits * off);
  rc |= n->alloc(&n->lpart, (size_t)nblk(E, 4) + 3 * (size_t)nblk(C, 4));
  rc |= n->alloc(&n->loss_out, 4);
  rc |= n->alloc(&n->mpart, 2 * (size_t)nblk(C, 4));
  rc |= n->alloc(&n->shift, 1);
  rc |= n->alloc(&n->checks, 4);
  rc |= n->alloc(&n->cpart, 3 * (size_t)nblk(C, 4));
  rc |= n->alloc(&n->mass_out, 1);
  if (rc) {
    *err = "device allocation for the corrector failed";
    delete n;
    return nullptr;
  }
  return n;
}

void destroy(Net *n) { delete n; }
size_t param_count(const Net *n) { return n->n_params; }

int set_params(Net &n, const float *host, hipStream_t s) {
  if (hipMemcpyAsync(n.params, host, n.n_params * sizeof(float), hipMemcpyHostToDevice, s) != hipSuccess) return -1;
  if (hipMemsetAsync(n.adam_m, 0, n.n_params * sizeof(float), s) != hipSuccess) return -1;
  if (hipMemsetAsync(n.adam_v, 0, n.n_params * sizeof(float), s) != hipSuccess) return -1;
  if (sync_bf16(n, s)) return -1;
  return hipStreamSynchronize(s) == hipSuccess ? 0 : -1;
}

int get_vec(const Net &n, int which, float *host, hipStream_t s) {
  const float *src = which == 0 ? n.params : n.grads;
  if (hipMemcpyAsync(host, src, n.n_params * sizeof(float), hipMemcpyDeviceToHost, s) != hipSuccess) return -1;
  return hipStreamSynchronize(s) == hipSuccess ? 0 : -1;
}

int set_scales(Net &n, const float *in_mean, const float *in_scale, const float *out_scale, hipStream_t s) {
  if (hipMemcpyAsync(n.in_mean, in_mean, KIN * sizeof(float), hipMemcpyHostToDevice, s) != hipSuccess ||
      hipMemcpyAsync(n.in_scale, in_scale, KIN * sizeof(float), hipMemcpyHostToDevice, s) != hipSuccess ||
      hipMemcpyAsync(n.out_scale, out_scale, NOUT * sizeof(float), hipMemcpyHostToDevice, s) != hipSuccess)
    return -1;
  return hipStreamSynchronize(s) == hipSuccess ? 0 : -1;
}

int raw_features(Net &n, const Instance &I, const int *old_c, float *dst, hipStream_t s) {
  if (!n.raw && n.alloc(&n.raw, (size_t)n.C * KIN)) return -1;
  if (features(n, I, s, n.raw)) return -1;
  hipLaunchKernelGGL(k_export_rows, dim3(nblk((size_t)n.C * KIN)), dim3(256), 0, s, (const float *)n.raw, old_c, n.C,
                     KIN, dst);
  return hipGetLastError() == hipSuccess ? 0 : -1;
}

int export_buf(Net &n, int what, const int *old_c, const int *old_e, float *dst, hipStream_t s) {
  switch (what) {
    case HEXDYN_NET_X:
      hipLaunchKernelGGL(k_export_rows_bf16, dim3(nblk((size_t)n.C * KIN)), dim3(256), 0, s, (const bf16 *)n.X, old_c,
                         n.C, KIN, dst);
      break;
    case HEXDYN_NET_Y:
      hipLaunchKernelGGL(k_export_rows, dim3(nblk((size_t)n.C * NOUT)), dim3(256), 0, s, (const float *)n.Y, old_c,
                         n.C, NOUT, dst);
      break;
    case HEXDYN_NET_TARGET_CELLS:
      hipLaunchKernelGGL(k_export_rows, dim3(nblk((size_t)n.C * 3 * HX_ROW)), dim3(256), 0, s, (const float *)n.Tc,
                         old_c, n.C, 3 * HX_ROW, dst);
      break;
    case HEXDYN_NET_TARGET_EDGES:
      hipLaunchKernelGGL(k_export_rows, dim3(nblk((size_t)n.E * HX_ROW)), dim3(256), 0, s, (const float *)n.Te, old_e,
                         n.E, HX_ROW, dst);
      break;
    default:
      return 1;
  }
  return hipGetLastError() == hipSuccess ? 0 : -1;
}

}  // namespace net
}  // namespace hexdyn
