/*
 * FP64 global integrals of the published state: dry mass, rho*theta_m,
 * total energy and the tracer masses, each a sum over cells and levels with
 * the cell-volume weight areaCell * dzw in binary64.
 *
 * The weights and products are formed in binary64 from the binary32 fields
 * (the reference's owned-union totals, cuda_fullstep_lts_active.py:1337-1360,
 * sum rho * (area * dzw) in float64 the same way).  Reduction order is fixed:
 * a lane tree inside each cell row, the block's four rows in order, then one
 * block sums the per-block partials in contiguous chunks with Neumaier
 * compensation and a fixed tree over the chunks.  Repeated calls on the same
 * state return identical bits.
 *
 * Total energy density: rho_zz * (c_v T + g z + K), T = theta_m * exner /
 * (1 + (R_v/R_d) q_v) with q_v the first scalar when the state is moist, z the
 * layer-mid height from zgrid (no potential term without zgrid), K the cell
 * kinetic energy (1/A) sum_e dc dv u_e^2 / 4.
 */
#include <hip/hip_runtime.h>

#include "hexdyn_internal.h"

namespace hexdyn {
namespace {

constexpr double kCv = 1004.5 - 287.0;
constexpr double kG = 9.80616;
constexpr double kRvRd = 461.6 / 287.0;

struct IntegralArgs {
  const float *rho, *rt, *q, *theta, *exner, *u;
  const float *zmid;   // [C][64] layer-mid heights (may be null)
  int NT, moist;
};

// Value of lane i + OFF, where the tree below needs it (lanes below OFF):
// half-wave and row swaps, and shifts inside a row of 16.
template <int OFF>
__device__ __forceinline__ unsigned down(unsigned v) {
  if constexpr (OFF == 32) return __builtin_amdgcn_permlane32_swap(v, v, false, false)[1];
  if constexpr (OFF == 16) return __builtin_amdgcn_permlane16_swap(v, v, false, false)[1];
  if constexpr (OFF < 16) return __builtin_amdgcn_update_dpp(v, v, 0x100 + OFF, 0xf, 0xf, false);  // row_shl
}
template <int OFF>
__device__ __forceinline__ void add_down(double &x) {
  const unsigned long long u = __double_as_longlong(x);
  const unsigned lo = down<OFF>((unsigned)u), hi = down<OFF>((unsigned)(u >> 32));
  x += __longlong_as_double(((unsigned long long)hi << 32) | lo);
}
// fixed-order tree over the 64 lanes of each of N values; lane 0 holds the
// totals.  Through the LDS permute unit the exchanges, twelve a value, held up
// the CU: all integrals of x1.40962 86.5 -> 71.3 us.
template <int N>
__device__ __forceinline__ void wave_sums(double (&x)[N]) {
#pragma unroll
  for (int i = 0; i < N; ++i) {
    add_down<32>(x[i]);
    add_down<16>(x[i]);
    add_down<8>(x[i]);
    add_down<4>(x[i]);
    add_down<2>(x[i]);
    add_down<1>(x[i]);
  }
}

// Species whose rows are loaded together.
constexpr int IQ = 6;

// Four cells a block, one wavefront each.  Blocks are renumbered so that an
// XCD owns a contiguous range of cells (the same edges' rows in its L2), and
// the rows a wavefront needs, the species' too, are loaded before the first
// sum: each sum is a chain of lane exchanges, and a species' load behind the
// sum before it is one more round trip.  26.9 -> 21.9 us at x1.10242 with six
// species, 17.8 with the sums' exchanges in registers.  A group is summed whole,
// species past the last one too: a call with its wait takes 33.2, 37.9 and 42.8 us
// for one, six and seven species there (52.6, 73.8 and 77.1 with one species after
// another, their exchanges through the permute unit).
template <int NE>
__global__ void __launch_bounds__(256) k_integrals(const Instance I, const IntegralArgs a, double *partial) {
  extern __shared__ double s_part[];  // [4 waves][NQ]
  const int NQ = 3 + a.NT;
  const int w = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const int nb = gridDim.x, x = blockIdx.x & 7, j = blockIdx.x >> 3, per = nb >> 3, rest = nb & 7;
  const int lb = x < rest ? x * (per + 1) + j : rest * (per + 1) + (x - rest) * per + j;
  const int c0 = lb * 4 + w;
  const int k = (int)(threadIdx.x & 63);
  const bool live = c0 < I.n.C && k < I.n.L;
  const int c = c0 < I.n.C ? c0 : 0;
  const int rs = I.n.RS;
  const size_t row = (size_t)c * rs + (k < rs ? k : rs - 1);  // rows rs floats apart
  const int n = I.m.neoc[c];
  float ue[NE], dd[NE], q[IQ];
#pragma unroll
  for (int s = 0; s < NE; ++s) {
    const int e = I.m.eoc[c * NE + s];
    ue[s] = a.u[(size_t)e * rs + (k < rs ? k : rs - 1)];
    dd[s] = I.m.dcdv[e];
  }
#pragma unroll
  for (int i = 0; i < IQ; ++i) q[i] = i < a.NT ? a.q[(size_t)i * I.n.C * rs + row] : 0.0f;
  const float rhof = a.rho[row], rtf = a.rt[row], thf = a.theta[row], exf = a.exner[row];
  const double z = a.zmid ? (double)a.zmid[row] : 0.0;
  const float ia = I.m.invarea[c];
  double wgt = 0.0;
  double rho = 0.0;
  if (live) {
    wgt = (1.0 / (double)ia) * (1.0 / (double)I.z.rdzw[k]);
    rho = (double)rhof;
  }
  // kinetic energy at the cell centre
  double ke = 0.0;
#pragma unroll
  for (int s = 0; s < NE; ++s) {
    const double u = (double)ue[s];
    if (s < n) ke += 0.25 * (double)dd[s] * u * u;
  }
  ke *= (double)ia;
  double qv = 0.0;
  if (a.moist && a.NT > 0) qv = (double)q[0];
  const double temp = (double)thf * (double)exf / (1.0 + kRvRd * qv);
  double vals[3];
  vals[0] = wgt * rho;
  vals[1] = live ? wgt * (double)rtf : 0.0;
  vals[2] = live ? wgt * rho * (kCv * temp + kG * z + ke) : 0.0;
  wave_sums(vals);
  if (k == 0)
    for (int i = 0; i < 3; ++i) s_part[w * NQ + i] = vals[i];
  for (int sp0 = 0; sp0 < a.NT; sp0 += IQ) {
    if (sp0 > 0) {
#pragma unroll
      for (int i = 0; i < IQ; ++i)
        q[i] = sp0 + i < a.NT ? a.q[(size_t)(sp0 + i) * I.n.C * rs + row] : 0.0f;
    }
    double m[IQ];
#pragma unroll
    for (int i = 0; i < IQ; ++i) m[i] = live ? wgt * rho * (double)q[i] : 0.0;
    wave_sums(m);
    if (k == 0) {
#pragma unroll
      for (int i = 0; i < IQ; ++i)
        if (sp0 + i < a.NT) s_part[w * NQ + 3 + sp0 + i] = m[i];
    }
  }
  __syncthreads();
  if ((int)threadIdx.x < NQ) {
    const int i = (int)threadIdx.x;
    partial[(size_t)lb * NQ + i] = ((s_part[i] + s_part[NQ + i]) + s_part[2 * NQ + i]) + s_part[3 * NQ + i];
  }
}

// block i: quantity i of nb partials -> out[i] (device or host memory).  One
// block for all quantities ran them one after the other, each a chain of
// chunk loads and a tree of barriers: 24.7 -> 6.3 us at x1.10242 with six
// species.
__global__ void __launch_bounds__(256) k_integrals_final(const double *partial, int nb, int NQ, double *out) {
  __shared__ double s_sum[256];
  const int t = (int)threadIdx.x, i = (int)blockIdx.x;
  const int chunk = (nb + 255) / 256;
  double sum = 0.0, comp = 0.0;
  const int b0 = t * chunk, b1 = min(nb, b0 + chunk);
  for (int b = b0; b < b1; ++b) {
    const double x = partial[(size_t)b * NQ + i];
    const double tt = sum + x;
    comp += fabs(sum) >= fabs(x) ? (sum - tt) + x : (x - tt) + sum;  // Neumaier
    sum = tt;
  }
  s_sum[t] = sum + comp;
  __syncthreads();
  for (int off = 128; off >= 1; off >>= 1) {
    if (t < off) s_sum[t] = s_sum[t] + s_sum[t + off];
    __syncthreads();
  }
  if (t == 0) out[i] = s_sum[0];
}

}  // namespace

int integrals(const Instance &I, const float *rho, const float *rt, const float *q, const float *theta,
              const float *exner, const float *u, const float *zmid, double *partial, double *out,
              hipStream_t s) {
  IntegralArgs a{rho, rt, q, theta, exner, u, zmid, I.n.NT, I.n.NM > 0};
  const int nb = (I.n.C + 3) / 4;
  const int NQ = 3 + I.n.NT;
  const size_t shm = (size_t)4 * NQ * sizeof(double);
  if (I.n.ME == 6)
    hipLaunchKernelGGL(k_integrals<6>, dim3(nb), dim3(256), shm, s, I, a, partial);
  else
    hipLaunchKernelGGL(k_integrals<7>, dim3(nb), dim3(256), shm, s, I, a, partial);
  hipLaunchKernelGGL(k_integrals_final, dim3(NQ), dim3(256), 0, s, (const double *)partial, nb, NQ, out);
  return hipGetLastError() == hipSuccess ? 0 : -1;
}

}  // namespace hexdyn
