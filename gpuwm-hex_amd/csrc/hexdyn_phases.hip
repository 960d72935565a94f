/*
 * hexdyn device kernels and the phase functions that launch them.
 *
 * This translation unit is compiled twice: with -ffp-contract=off into
 * namespace hexdyn::strict (every binary32 multiply and add rounded
 * separately, in the reference's operand order, so results equal the CPU
 * restatement bit for bit) and with -ffp-contract=fast into hexdyn::fast.
 *
 * Mapping: a block of 256 threads is 4 wavefronts; each wavefront owns one
 * entity (cell, edge or vertex) row of 64 floats and lane k owns level k.
 * Connectivity of the entity is wave-uniform (scalar loads); neighbour rows
 * are read as whole 256-byte lines, so every cellsOnEdge / edgesOnCell /
 * advCellsForEdge gather is one coalesced access per neighbour.  Blocks are
 * renumbered so each XCD (hardware assigns block b to XCD b % 8) works on a
 * contiguous range of the space-filling-curve order and its L2 sees the
 * neighbour rows it needs.  Vertical neighbours come from cross-lane moves;
 * the serial column recurrences (Thomas sweep, implicit coefficients) pass
 * from lane to lane, in the reference's arithmetic order.
 *
 * Reference operators (operation order per element):
 *   solve diagnostics  cuda_horizontal_v841.py:67-200, diagnostics.py:95-306
 *   dyn tendencies     dynamics.py:86-268, dynamics_v841.py:128-185,
 *                      driver.py:933-1207, acoustic.py:246-281
 *   implicit coefs     acoustic_v841.py:81-233
 *   acoustic substep   acoustic_v841.py:296-565
 *   divergence damping mixing.py:851-945
 *   recovery           driver.py:3176-3290, driver.py:819-876, terrain.py:491-571
 *   scalar transport   transport.py:1649-1826, transport.py:1829-2175
 */
#include <hip/hip_runtime.h>

#include "hexdyn_div.h"
#include "hexdyn_internal.h"
#include "hexdyn_powf.h"

#ifndef HEXDYN_NS
#define HEXDYN_NS strict
#endif

namespace hexdyn {
namespace HEXDYN_NS {
namespace {

// Element k of row ent of p, addressed as a 32-bit byte offset from the
// wave-uniform base (every array is below 4 GiB), so loads and stores take
// the SGPR-base + VGPR-offset form instead of a per-lane 64-bit address.
// Rows are rs floats apart (the level count plus one, rounded up to 8:
// 224-byte rows at 55 levels, so a streamed array moves 12.5 % fewer bytes
// than with 64-float rows, while a gathered row still spans four 64-byte
// sectors).  Lanes k >= rs read the row's last element instead of the next
// row: for layer arrays that element is padding (zero), so every lane sees
// what a 64-float row would hold; for interface arrays it is the top value,
// which no lane at or below the top reads through a shuffle.  Stores are
// made for k <= L < rs only.
__device__ __forceinline__ uint32_t row_off(int rs, int ent, int k) {
  return (uint32_t)ent * (uint32_t)(rs * 4) + (uint32_t)(k < rs ? k : rs - 1) * 4u;
}
#define AT(p, ent, k) (*(float *)((char *)(p) + row_off(I.n.RS, (ent), (k))))
// gather kernels take up to 16 rows (wavefronts) per block: a per-kernel launch setting
#define KB __global__ void __launch_bounds__(1024)

// First entity of this block: blocks are renumbered so that XCD x (hardware
// block b runs on XCD b % 8) owns a contiguous range of the curve.  wpb is
// the number of wavefronts (entities) per block.
__device__ __forceinline__ int block_entity0(int b, int nb, int wpb) {
  const int x = b & 7, i = b >> 3, q = nb >> 3, r = nb & 7;
  const int lb = (x < r) ? x * (q + 1) + i : r * (q + 1) + (x - r) * q + i;
  return lb * wpb;
}
__device__ __forceinline__ int block_entity0(int wpb) { return block_entity0(blockIdx.x, gridDim.x, wpb); }
// Column kernels: WPB rows per block, fixed at compile time.
template <int WPB>
__device__ __forceinline__ int wave_entity() {
  return __builtin_amdgcn_readfirstlane(block_entity0(WPB) + (int)(threadIdx.x >> 6));
}
// Gather kernels: the block size is a per-kernel launch setting, carried in
// the kernel's own Instance argument (I.n.WPB) rather than read from the
// dispatch packet, which would cost each wavefront a vector-memory round trip
// before its first row load.
__device__ __forceinline__ int wave_entity(const Instance &I) {
  return __builtin_amdgcn_readfirstlane(block_entity0(I.n.WPB) + (int)(threadIdx.x >> 6));
}
// Two independent gather passes in one launch: the first nb0 blocks (a
// multiple of 8, so that the second pass's blocks keep their XCDs) are the
// first pass's, the others the second's.
__device__ __forceinline__ int wave_entity_first(const Instance &I, int nb0) {
  return __builtin_amdgcn_readfirstlane(block_entity0(blockIdx.x, nb0, I.n.WPB) + (int)(threadIdx.x >> 6));
}
__device__ __forceinline__ int wave_entity_second(const Instance &I, int nb0) {
  return __builtin_amdgcn_readfirstlane(block_entity0(blockIdx.x - nb0, gridDim.x - nb0, I.n.WPB) +
                                        (int)(threadIdx.x >> 6));
}
__device__ __forceinline__ int lane() { return (int)(threadIdx.x & 63); }
// Value of lane k-1 (lane 0: its own) and k+1 (lane 63: its own): whole-wave
// DPP shifts, one VALU move each.  The generic shuffles go through the LDS
// permute unit, a round trip that also waits for every scalar load in flight
// (four x1.40962 steps with their output: 24.41 -> 24.27 ms).
// Call with every lane active (outside lane-dependent branches).
__device__ __forceinline__ float up1(float x) {
  const int v = __float_as_int(x);
  return __int_as_float(__builtin_amdgcn_update_dpp(v, v, 0x138, 0xf, 0xf, false));  // wave_shr:1
}
__device__ __forceinline__ float dn1(float x) {
  const int v = __float_as_int(x);
  return __int_as_float(__builtin_amdgcn_update_dpp(v, v, 0x130, 0xf, 0xf, false));  // wave_shl:1
}
__device__ __forceinline__ float rdl(float x, int j) {
  return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(x), j));
}
__device__ __forceinline__ float cs1(float x) { return __builtin_copysignf(1.0f, x); }
__device__ __forceinline__ float max0(float x) { return x > 0.0f ? x : 0.0f; }
__device__ __forceinline__ float min0(float x) { return x < 0.0f ? x : 0.0f; }
__device__ __forceinline__ float pmin(float a, float b) { return b < a ? b : a; }
__device__ __forceinline__ float pmax(float a, float b) { return b > a ? b : a; }
// x / 12 with IEEE round-to-nearest.  For quotients in [2^-125, FLT_MAX] the
// product by RN(1/12) plus one FMA residual correction is the correctly
// rounded quotient (verified exhaustively over every binary32 x); zeros,
// tiny, infinite and NaN inputs take the division itself.
__device__ __forceinline__ float div12(float x) {
  constexpr float r12 = 0x1.555556p-4f;  // RN(1/12)
  const float q0 = x * r12;
  const float a = fabsf(q0);
  if (a >= 0x1p-125f && a <= 0x1.fffffep127f) return __builtin_fmaf(__builtin_fmaf(-q0, 12.0f, x), r12, q0);
  return x / 12.0f;
}

__device__ __forceinline__ float flux4(float qm2, float qm1, float q0, float qp1, float vel) {
  return div12(vel * (7.0f * (q0 + qm1) - (qp1 + qm2)));
}
__device__ __forceinline__ float flux3(float qm2, float qm1, float q0, float qp1, float vel, float coef) {
  return flux4(qm2, qm1, q0, qp1, vel) + div12((coef * fabsf(vel)) * ((qp1 - qm2) - 3.0f * (q0 - qm1)));
}

__device__ __forceinline__ void set_flag(int *flag) { atomicOr(flag, 1); }

// exner = arg^(R/cv) with the GNU powf bits the reference's v8.4.1 recovery
// uses (cuda_driver.py:1466-1472): the correctly rounded binary64 method,
// moved to the other neighbour where the host-built bitmap marks the argument.
__device__ __forceinline__ float exner_pow(const Instance &I, float arg) {
  const double d = hexdyn_pow_d(arg, I.k.rcv);
  return hexdyn_gnu_powf_fix(arg, (float)d, d, I.m.powf_ties, I.k.powf_near_tie);
}

// Per-slot coefficients of one entity (its row of N values in an [n][N]
// table), read by one vector load with lane s taking slot s and issued with
// the row loads; slot s is read from lane s where it is used.  The same
// values as scalar loads miss the scalar cache for every entity, and the
// compiler issues such loads next to their uses, after the rows have
// arrived, so each becomes a dependent round trip of the wavefront.
// Read a slot only in wave-uniform control flow: the compiler may move the
// load into the first branch that reads the row, and in a lane-divergent
// branch the lanes that hold the other slots would not execute it.  Code
// that needs slots under a lane condition takes them with slot_vals first.
template <int N>
struct SlotRow {
  float v;  // lane s: slot s
  __device__ __forceinline__ float operator[](int s) const { return rdl(v, s); }
};
template <int N>
__device__ __forceinline__ SlotRow<N> slot_row(const float *__restrict__ p) {
  const int l = lane();
  return {p[l < N ? l : N - 1]};
}
// every slot as a wave-uniform value (call with all lanes active)
template <int N>
__device__ __forceinline__ void slot_vals(SlotRow<N> &r, float (&o)[N]) {
#pragma unroll
  for (int s = 0; s < N; ++s) o[s] = r[s];
}
// Ends the load phase for x: the compiler may not sink the load of x into
// the first (uniform) branch that uses it, which would issue it, and the
// scalar index load it needs, one round trip after the others.
__device__ __forceinline__ void keep(float &x) { asm volatile("" : "+v"(x)); }
template <int N>
__device__ __forceinline__ void keep(float (&x)[N]) {
#pragma unroll
  for (int i = 0; i < N; ++i) keep(x[i]);
}
template <int G, int N>
__device__ __forceinline__ void keep(float (&x)[G][N]) {
#pragma unroll
  for (int g = 0; g < G; ++g) keep(x[g]);
}
template <class... T>
__device__ __forceinline__ void keep(T &...x) {
  (keep(x), ...);
}
// Marks slot rows as read only after this point: called once the
// wavefront's row loads are issued, so the lane reads of the slots (which
// wait for the slot loads) are not scheduled ahead of the row loads.  Call
// with all lanes active.  Emits nothing.
template <class R>
__device__ __forceinline__ void settle1(R &row) {
  asm volatile("" : "+v"(row.v));
}
template <class... R>
__device__ __forceinline__ void settle(R &...rows) {
  (settle1(rows), ...);
}
// Ends the index phase of a wavefront: every scalar index load issued before
// the first fence completes in one wait, before any row load after it is
// issued.  Without it the compiler may issue one index table's loads only
// after waiting for another's, one more dependent round trip.
__device__ __forceinline__ void fence(int x) { asm volatile("" ::"s"(x)); }
// Loads after this point are issued after it (a pass in several parts holds
// back the rows of the next part, whose registers the part before frees).
__device__ __forceinline__ void hold_loads() { asm volatile("" ::: "memory"); }
// A per-entity value read by a vector load (every lane the same address) for
// the same reason; the zero offset is opaque, so the load stays a vector load.
__device__ __forceinline__ float uni_load(const float *__restrict__ p) {
  int z;
  asm("v_mov_b32 %0, 0" : "=v"(z));
  return p[z];
}

inline int nblocks(int n, int wpb) { return (n + wpb - 1) / wpb; }

// Column kernels: W cells (one wavefront each) per block, which share the
// per-level coefficient rows in LDS.  The implicit coefficients on their own
// take 16 columns per block, the acoustic column update and a stage's whole column
// pass 4 (a x1.40962 step with 2, 4 and 8 columns: 5049, 5030 and 5042 us).
constexpr int COLW_VC = 16;  // k_vcoef
constexpr int COLW_AC = 4;   // k_ac_cell and k_col
// Registers of k_vcoef and k_ac_cell for 8 wavefronts per SIMD: at 7 a CU would
// hold one block of 16 columns instead of two, and the acoustic update at 6 takes
// 87 us for 82 (x1.40962).
#define KBCOL(W) __global__ void __launch_bounds__(64 * (W)) __attribute__((amdgpu_waves_per_eu(8, 8)))

// Per-level coefficient rows are the same for every column of a block: wave
// j < N of a column block copies row j into LDS once, instead of each of the
// 16 wavefronts reading every row.  Callers synchronise before reading.
template <int N>
__device__ __forceinline__ void stage_levels(float *s_lev, const float *const (&rows)[N], int w, int k) {
#pragma unroll
  for (int j = 0; j < N; ++j)
    if (w == j) s_lev[j * 64 + k] = rows[j][k];
}

// Value of lane k-1 (lane 0: zero) and k+1 (lane 63: zero): whole-wave DPP
// shifts that the compiler folds into the multiplication that reads them.
__device__ __forceinline__ float up0(float x) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), 0x138, 0xf, 0xf, true));
}
__device__ __forceinline__ float dn0(float x) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), 0x130, 0xf, 0xf, true));
}

// The serial recurrences of a column, lane k being level k: every lane repeats
// its level's step from its neighbour's last value, so after i steps the first
// i levels are final, and a further step gives them the same bits (the count
// rounds up to whole unrolled blocks; a lane exchange keeps the compiler from
// unrolling a loop with a remainder).  The dependent chain of a level is what
// one lane per column would run, which bounds the pass on small meshes; with
// one wavefront sweeping the columns of its block out of LDS the chain also
// waited for LDS reads and two block barriers, and the block's other
// wavefronts for it.  The issue slots are about the same, one column's steps
// on a whole wavefront against four columns' LDS reads and writes.  k_col with
// coefficients 12.1 -> 9.2 us and without 8.4 -> 6.9 at x1.162, k_ac_cell 8.8
// -> 8.1; at x1.40962, where other columns hide the chain, 96 + 115 + 94 -> 95
// + 112 + 93 us the stages of a subcycle.
// Thomas sweeps (acoustic_v841.py:296-565): forward for levels 1..L-1 with
// the sub-diagonal d and 1/denominator l, back substitution with g for levels
// L-1..0.  Levels past L give zero.
__device__ __forceinline__ float thomas_sweeps(float x, float d, float l, float g, int k, int L) {
  const bool inner = k >= 1 && k < L;
  d = inner ? d : 0.0f;
  l = inner ? l : 1.0f;
  g = inner ? g : 0.0f;
  x = k <= L ? x : 0.0f;
  float p = x;
  for (int i = 1; i < L; i += 8) {
#pragma unroll
    for (int u = 0; u < 8; ++u) p = (x - d * up0(p)) * l;
  }
  p = x = inner ? p : x;  // level L's 0 * (a value that is not finite) stays out
  for (int i = 0; i < L; i += 8) {
#pragma unroll
    for (int u = 0; u < 8; ++u) p = x - g * dn0(p);
  }
  return p;
}
// alpha/gamma recurrence up the column (acoustic_v841.py:81-233): alpha over
// a, gamma over b, zero at the levels that have no equation; returns 1 where
// this level's denominator vanishes.  With the corrected reciprocal, and where
// one of the column's final denominators left that one's range again with the
// division.
__device__ __forceinline__ int coef_sweep(float &a, float &b, float c, int k, int L, float dts2) {
  const bool inner = k >= 1 && k < L;
  a = inner ? a : 0.0f;
  b = inner ? b : 0.0f;
  c = inner ? dts2 * c : 0.0f;
  float gm = 0.0f, al = 1.0f, den = 1.0f;
  for (int i = 1; i < L; i += 8) {  // L - 1 steps in whole blocks
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      den = 1.0f + dts2 * (b - a * up0(gm));
      al = recip(den);
      gm = c * al;
    }
  }
  int singular = 0;
  if (__any(!recip_in_range(den))) {
    gm = 0.0f;
    for (int i = 1; i < L; ++i) {
      den = 1.0f + dts2 * (b - a * up0(gm));
      al = 1.0f / den;
      gm = c * al;
    }
    singular = den == 0.0f ? 1 : 0;
  }
  a = inner ? al : 0.0f;
  b = inner ? gm : 0.0f;
  return singular;
}

// Gather helpers.  Connectivity rows are padded to fixed widths (NE = maxEdges
// slots per cell, NX = 2*maxEdges-2 slots per edge) with index 0, so every
// slot of an unrolled loop addresses a valid row.  All neighbour rows are
// loaded before any arithmetic, then combined in slot order for the valid
// slots only, which keeps the reference's association and lets the memory
// system overlap every gather of the wave.

// ------------------------------------------------------------------ diagnostics
KB k_diag_vertex(const Instance I, const float *__restrict__ u, int store_mix) {
  const int v = wave_entity(I);
  if (v >= I.n.V) return;
  const int k = lane();
  int e[3];
  float ue[3];
#pragma unroll
  for (int s = 0; s < 3; ++s) e[s] = I.m.eov[3 * v + s];
  SlotRow<3> dc = slot_row<3>(I.m.vdc + 3 * v), dcdv = slot_row<3>(I.m.vdcdv + 3 * v);
  const float it = uni_load(I.m.invtri + v), fv = uni_load(I.m.fvert + v);
#pragma unroll
  for (int s = 0; s < 3; ++s) fence(e[s]);
#pragma unroll
  for (int s = 0; s < 3; ++s) ue[s] = AT(u, e[s], k);
  keep(ue, it, fv);
  settle(dc, dcdv);
  float vort = 0.0f, kev = 0.0f;
#pragma unroll
  for (int s = 0; s < 3; ++s) {
    vort = vort + dc[s] * ue[s];
    kev = kev + dcdv[s] * (ue[s] * ue[s]);
  }
  vort = vort * it;
  kev = kev * (0.25f * it);
  const float pvv = fv + vort;
  if (k < I.n.L) {
    if (store_mix) AT(I.b.vorticity, v, k) = vort;
    AT(I.b.ke_vertex, v, k) = kev;
    AT(I.b.pv_vertex, v, k) = pvv;
  }
}

// divergence, kinetic energy (0.625/0.375 kite blend) and pv_cell of cell c
struct CellDiag {
  float div, ke, pv;
};
template <int NE>
struct CellDiagIn {
  float ue[NE], kv[NE], pv[NE];
  SlotRow<NE> sd, dd, kt;
  float ia;
  int n;
};
template <int NE>
__device__ __forceinline__ CellDiagIn<NE> diag_cell_load(const Instance &I, const float *__restrict__ u, int c,
                                                         int k) {
  CellDiagIn<NE> a;
  a.n = I.m.neoc[c];
  int e[NE], vv[NE];
#pragma unroll
  for (int s = 0; s < NE; ++s) {
    e[s] = I.m.eoc[c * NE + s];
    vv[s] = I.m.voc[c * NE + s];
  }
  a.sd = slot_row<NE>(I.m.csdv + c * NE);
  a.dd = slot_row<NE>(I.m.cdcdv + c * NE);
  a.kt = slot_row<NE>(I.m.ckite + c * NE);
  a.ia = uni_load(I.m.invarea + c);
#pragma unroll
  for (int s = 0; s < NE; ++s) {
    fence(e[s]);
    fence(vv[s]);
  }
#pragma unroll
  for (int s = 0; s < NE; ++s) {
    a.ue[s] = AT(u, e[s], k);
    a.kv[s] = AT(I.b.ke_vertex, vv[s], k);
    a.pv[s] = AT(I.b.pv_vertex, vv[s], k);
  }
  keep(a.ue, a.kv, a.pv, a.ia);
  settle(a.sd, a.dd, a.kt);
  return a;
}
template <int NE>
__device__ __forceinline__ CellDiag diag_cell_compute(const Instance &I, const CellDiagIn<NE> &a) {
  const int n = a.n;
  const float ia = a.ia;
  float d = 0.0f, kc = 0.0f, pvc = 0.0f;
#pragma unroll
  for (int s = 0; s < NE; ++s)
    if (s < n) {
      d = d + a.sd[s] * a.ue[s];
      kc = kc + 0.25f * (a.dd[s] * (a.ue[s] * a.ue[s]));
    }
  d = d * ia;
  kc = kc * ia;
  kc = kc * 0.625f;
#pragma unroll
  for (int s = 0; s < NE; ++s)
    if (s < n) {
      const float kite = a.kt[s];
      float corr = 0.375f * kite;
      corr = corr * a.kv[s];
      corr = corr * ia;
      kc = kc + corr;
      pvc = pvc + (kite * a.pv[s]) * ia;
    }
  return {d, kc, pvc};
}
__device__ __forceinline__ void store_cell_diag(const Instance &I, int c, int k, CellDiag r, int store_mix) {
  if (k < I.n.L) {
    if (store_mix) AT(I.b.divergence, c, k) = r.div;
    AT(I.b.ke, c, k) = r.ke;
    if (I.k.apvm_on) AT(I.b.pv_cell, c, k) = r.pv;
  }
}

template <int NE>
KB k_diag_cell(const Instance I, const float *__restrict__ u, int store_mix) {
  const int c = wave_entity(I);
  if (c >= I.n.C) return;
  const int k = lane();
  store_cell_diag(I, c, k, diag_cell_compute<NE>(I, diag_cell_load<NE>(I, u, c, k)), store_mix);
}

// The same, with the vertices of the cell formed here from the cell's edges and
// each vertex's third edge instead of in a pass of their own (Sizes::VP): 12
// u rows a cell in place of 6 u and 12 vertex rows, and no vertex pass (6 u
// rows and 4 stores a cell): 33.8 us against 26.3 + 18.8 at x1.40962.  The
// owning cell stores the vertex's
// pv_vertex (and vorticity for the mixing).  A vertex's three terms are added
// in edgesOnVertex order; its first two commute, so of the cell's edges P (slot
// s) and Q (slot s - 1) and the third edge X the code names the last, and the
// record holds the weights in that order.
template <int NE>
struct CellVertIn {
  float uo[NE], ux[NE];
  SlotRow<NE> sd, dd, kt;
  SlotRow<HX_ROW> rec;
  float ia;
  int n, code, e[NE], x[NE], v[NE];
};
template <int NE>
__device__ __forceinline__ void cell_vert_index(const Instance &I, int c, CellVertIn<NE> &a) {
  a.n = I.m.neoc[c];
  a.code = I.m.vcode[c];
#pragma unroll
  for (int s = 0; s < NE; ++s) {
    a.e[s] = I.m.eoc[c * NE + s];
    a.x[s] = I.m.vx[c * NE + s];
    a.v[s] = I.m.voc[c * NE + s];
  }
  a.sd = slot_row<NE>(I.m.csdv + c * NE);
  a.dd = slot_row<NE>(I.m.cdcdv + c * NE);
  a.kt = slot_row<NE>(I.m.ckite + c * NE);
  a.rec = slot_row<HX_ROW>(I.m.vrec + c * HX_ROW);
  a.ia = uni_load(I.m.invarea + c);
}
template <int NE>
__device__ __forceinline__ void cell_vert_fence(const CellVertIn<NE> &a) {
  fence(a.code);
#pragma unroll
  for (int s = 0; s < NE; ++s) {
    fence(a.e[s]);
    fence(a.x[s]);
    fence(a.v[s]);
  }
}
template <int NE>
__device__ __forceinline__ void cell_vert_rows(const Instance &I, const float *__restrict__ u, int k,
                                               CellVertIn<NE> &a) {
#pragma unroll
  for (int s = 0; s < NE; ++s) {
    a.uo[s] = AT(u, a.e[s], k);
    a.ux[s] = AT(u, a.x[s], k);
  }
}
template <int NE>
__device__ __forceinline__ void cell_vert_finish(const Instance &I, int c, int k, const CellVertIn<NE> &a,
                                                 int store_mix) {
  const int n = a.n, L = I.n.L;
  float d = 0.0f, kc = 0.0f, pvc = 0.0f;
#pragma unroll
  for (int s = 0; s < NE; ++s)
    if (s < n) {
      d = d + a.sd[s] * a.uo[s];
      kc = kc + 0.25f * (a.dd[s] * (a.uo[s] * a.uo[s]));
    }
  d = d * a.ia;
  kc = kc * a.ia;
  kc = kc * 0.625f;
  float uq = a.uo[2];  // the edge row of slot s - 1: of the last slot for s = 0
#pragma unroll
  for (int s = 3; s < NE; ++s) uq = s < n ? a.uo[s] : uq;
#pragma unroll
  for (int s = 0; s < NE; ++s)
    if (s < n) {
      const float up = a.uo[s], ux = a.ux[s];
      const int r = s * HX_VREC, last = a.code >> (2 * s) & 3;
      const float u0 = last == 0 ? uq : up, u1 = last == 2 ? uq : ux, u2 = last == 2 ? ux : last == 1 ? uq : up;
      const float it = a.rec[r + 6], fv = a.rec[r + 7];
      float vort = 0.0f + a.rec[r] * u0;
      vort = vort + a.rec[r + 1] * u1;
      vort = vort + a.rec[r + 2] * u2;
      vort = vort * it;
      float kev = 0.0f + a.rec[r + 3] * (u0 * u0);
      kev = kev + a.rec[r + 4] * (u1 * u1);
      kev = kev + a.rec[r + 5] * (u2 * u2);
      kev = kev * (0.25f * it);
      const float pvv = fv + vort;
      const float kite = a.kt[s];
      float corr = 0.375f * kite;
      corr = corr * kev;
      corr = corr * a.ia;
      kc = kc + corr;
      pvc = pvc + (kite * pvv) * a.ia;
      if (a.code >> (16 + s) & 1) {
        const int v = a.v[s];
        if (k < L) {
          AT(I.b.pv_vertex, v, k) = pvv;
          if (store_mix) AT(I.b.vorticity, v, k) = vort;
        }
      }
      uq = up;
    }
  store_cell_diag(I, c, k, {d, kc, pvc}, store_mix);
}
template <int NE>
KB k_diag_cv(const Instance I, const float *__restrict__ u, int store_mix) {
  const int c = wave_entity(I);
  if (c >= I.n.C) return;
  const int k = lane();
  CellVertIn<NE> a;
  cell_vert_index(I, c, a);
  cell_vert_fence(a);
  cell_vert_rows(I, u, k, a);
  keep(a.uo, a.ux, a.ia);
  settle(a.sd, a.dd, a.kt, a.rec);
  cell_vert_finish(I, c, k, a, store_mix);
}

// pv_edge (with APVM) and, at rk step 3, the TRiSK tangential velocity v of
// edge e.  The bodies below only load and compute; kernels store afterwards,
// so no load of a pass waits behind one of its own stores.
struct EdgeDiag {
  float v, pv;
};
template <int NE, bool RECON>
struct EdgeDiagIn {
  float un[RECON ? 2 * NE - 2 : 1];
  SlotRow<2 * NE - 2> wt;
  float vrow, pv0, pv1, pc0, pc1, ue, idv, idc;
  int n;
  int v0, v1, c0, c1, nb[RECON ? 2 * NE - 2 : 1];  // scalar index loads
};
// first phase: indices, slot counts and per-edge coefficients (none of
// which needs another load first)
template <int NE, bool RECON>
__device__ __forceinline__ void diag_edge_index(const Instance &I, int e, EdgeDiagIn<NE, RECON> &a) {
  constexpr int NX = 2 * NE - 2;
  a.v0 = I.m.voe[2 * e];
  a.v1 = I.m.voe[2 * e + 1];
  a.c0 = I.m.coe[2 * e];
  a.c1 = I.m.coe[2 * e + 1];
  a.idv = uni_load(I.m.invdv + e);
  a.idc = uni_load(I.m.invdc + e);
  if (RECON) {
#pragma unroll
    for (int s = 0; s < NX; ++s) a.nb[s] = I.m.eoe[e * NX + s];
    a.n = I.m.neoe[e];
    a.wt = slot_row<NX>(I.m.woe + e * NX);
  } else {
    a.wt = {0.0f};
    a.n = 0;
  }
}
template <int NE, bool RECON>
__device__ __forceinline__ void diag_edge_fence(const EdgeDiagIn<NE, RECON> &a) {
  fence(a.v0);
  fence(a.v1);
  fence(a.c0);
  fence(a.c1);
  if (RECON) {
#pragma unroll
    for (int s = 0; s < 2 * NE - 2; ++s) fence(a.nb[s]);
  }
}
// second phase: the rows (pv_cell and u are read whether or not APVM is on:
// both buffers always exist)
template <int NE, bool RECON>
__device__ __forceinline__ void diag_edge_rows(const Instance &I, const float *__restrict__ u, int e, int k,
                                               EdgeDiagIn<NE, RECON> &a) {
  constexpr int NX = 2 * NE - 2;
  if (RECON) {
#pragma unroll
    for (int s = 0; s < NX; ++s) a.un[s] = AT(u, a.nb[s], k);
    a.vrow = 0.0f;
  } else {
    a.vrow = AT(I.b.v, e, k);
  }
  a.pv0 = AT(I.b.pv_vertex, a.v0, k);
  a.pv1 = AT(I.b.pv_vertex, a.v1, k);
  a.pc0 = AT(I.b.pv_cell, a.c0, k);
  a.pc1 = AT(I.b.pv_cell, a.c1, k);
  a.ue = AT(u, e, k);
}
template <int NE, bool RECON>
__device__ __forceinline__ EdgeDiagIn<NE, RECON> diag_edge_load(const Instance &I, const float *__restrict__ u, int e,
                                                                int k) {
  EdgeDiagIn<NE, RECON> a;
  diag_edge_index(I, e, a);
  diag_edge_fence(a);
  diag_edge_rows(I, u, e, k, a);
  settle(a.wt);
  return a;
}
template <int NE, bool RECON>
__device__ __forceinline__ EdgeDiag diag_edge_compute(const Instance &I, int e, const EdgeDiagIn<NE, RECON> &a) {
  constexpr int NX = 2 * NE - 2;
  float vv;
  if (RECON) {
    vv = 0.0f;
#pragma unroll
    for (int s = 0; s < NX; ++s)
      if (s < a.n) vv = vv + a.wt[s] * a.un[s];
  } else {
    vv = a.vrow;
  }
  const float pve = 0.5f * (a.pv0 + a.pv1);
  // computed either way (a select, not a branch, so the loads are not sunk)
  const float gt = (a.pv1 - a.pv0) * a.idv;
  const float gn = (a.pc1 - a.pc0) * a.idc;
  const float pva = pve - I.k.apvm_scale * (vv * gt + a.ue * gn);
  return {vv, I.k.apvm_on ? pva : pve};
}
template <int NE, bool RECON>
__device__ __forceinline__ EdgeDiag diag_edge_values(const Instance &I, const float *__restrict__ u, int e, int k) {
  return diag_edge_compute<NE, RECON>(I, e, diag_edge_load<NE, RECON>(I, u, e, k));
}
__device__ __forceinline__ void store_edge_diag(const Instance &I, int e, int k, bool recon, EdgeDiag d) {
  if (k < I.n.L) {
    if (recon) AT(I.b.v, e, k) = d.v;
    AT(I.b.pv_edge, e, k) = d.pv;
  }
}

// RECON: rk step 3, where v is reconstructed (cuda_horizontal_v841.py:1058-1097)
template <int NE, bool RECON>
KB k_diag_edge(const Instance I, const float *__restrict__ u) {
  const int e = wave_entity(I);
  if (e >= I.n.E) return;
  const int k = lane();
  store_edge_diag(I, e, k, RECON, diag_edge_values<NE, RECON>(I, u, e, k));
}

// theta and w edge fluxes of a stage (defined with the tendencies)
struct EdgeFlux {
  float th, corr, w;
};
template <int NE>
struct EdgeFluxIn;
template <int NE, bool CORR>
__device__ __forceinline__ void tend_flux_index(const Instance &I, int e, int k, EdgeFluxIn<NE> &b);
template <int NE>
__device__ __forceinline__ void tend_flux_fence(const EdgeFluxIn<NE> &b);
template <int NE, bool CORR>
__device__ __forceinline__ void tend_flux_rows(const Instance &I, int e, int k, EdgeFluxIn<NE> &b);
template <int NE, bool CORR>
__device__ __forceinline__ EdgeFlux tend_flux_compute(const Instance &I, int e, const EdgeFluxIn<NE> &b);
template <bool CORR>
__device__ __forceinline__ void store_edge_flux(const Instance &I, int e, int k, EdgeFlux f);

// the edge diagnostics and, in the same pass, the next stage's theta/w edge
// fluxes: every input of those fluxes (theta, w, ru after recovery; the
// subcycle-start ru and theta) is final once recovery has run.  After rk
// step 3 (RECON) the next stage is a first stage (no RK correction flux);
// after rk steps 1 and 2 it is stage 2 or 3 (with the correction).
template <int NE, bool RECON>
KB k_diag_edge_flux(const Instance I, const float *__restrict__ u) {
  const int e = wave_entity(I);
  if (e >= I.n.E) return;
  const int k = lane();
  EdgeDiagIn<NE, RECON> a;
  EdgeFluxIn<NE> b;
  diag_edge_index(I, e, a);
  tend_flux_index<NE, !RECON>(I, e, k, b);
  diag_edge_fence(a);
  tend_flux_fence(b);
  diag_edge_rows(I, u, e, k, a);
  tend_flux_rows<NE, !RECON>(I, e, k, b);
  keep(b.thn, b.wn, b.rue, b.sru, b.sth0, b.sth1, b.fzm, b.fzp, b.dv);
  keep(a.un, a.vrow, a.pv0, a.pv1, a.pc0, a.pc1, a.ue, a.idv, a.idc);
  settle(a.wt, b.av, b.a3v);
  const EdgeDiag d = diag_edge_compute<NE, RECON>(I, e, a);
  const EdgeFlux f = tend_flux_compute<NE, !RECON>(I, e, b);
  store_edge_diag(I, e, k, RECON, d);
  store_edge_flux<!RECON>(I, e, k, f);
}

// The same pass over a tile of HX_TILE_E edges, one wavefront each: the
// theta and w rows of the tile's distinct advection cells cross the texture
// path once per tile into LDS, and the ten-cell stencils read them there.
// The gathers are bound by the texture path's rate per row load (about ten
// cycles per 256-byte row per CU), and consecutive edges along the curve
// share most stencil cells (about 2.8 distinct cells per edge instead of 10).
template <int NE, bool RECON>
__global__ void __launch_bounds__(64 * HX_TILE_E) k_diag_edge_flux_t(const Instance I, const float *__restrict__ u) {
  constexpr int NX = 2 * NE - 2, J = (HX_TILE_U + HX_TILE_E - 1) / HX_TILE_E;
  constexpr bool CORR = !RECON;
  __shared__ float s_th[HX_TILE_U * 64], s_w[HX_TILE_U * 64];
  const int w = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)), k = lane();
  const int tile = block_entity0(1);
  const int e0 = tile * HX_TILE_E + w;
  const bool live = e0 < I.n.E;
  const int e = live ? e0 : I.n.E - 1;  // every wavefront stages its share and reaches the barrier
  const int ncell = I.m.ntcell[tile];
  EdgeDiagIn<NE, RECON> a;
  EdgeFluxIn<NE> b;
  diag_edge_index(I, e, a);
  b.c0 = I.m.coe[2 * e];
  b.c1 = I.m.coe[2 * e + 1];
#pragma unroll
  for (int sl = 0; sl < NX; ++sl) b.ac[sl] = I.m.advl[e * NX + sl];  // slot -> row of the tile's cell list
  b.na = I.m.nadv[e];
  b.av = slot_row<NX>(I.m.adv + e * NX);
  b.a3v = slot_row<NX>(I.m.adv3 + e * NX);
  b.dv = CORR ? uni_load(I.m.dv + e) : 0.0f;
  b.fzm = AT(I.z.fzm, 0, k);
  b.fzp = AT(I.z.fzp, 0, k);
  int cr[J];
#pragma unroll
  for (int j = 0; j < J; ++j) cr[j] = I.m.tcell[tile * HX_TILE_U + min(w + j * HX_TILE_E, HX_TILE_U - 1)];
  diag_edge_fence(a);
  fence(b.c0);
  fence(b.c1);
#pragma unroll
  for (int j = 0; j < J; ++j) fence(cr[j]);
  float st[J], sw[J];
#pragma unroll
  for (int j = 0; j < J; ++j) {
    st[j] = sw[j] = 0.0f;
    if (w + j * HX_TILE_E < ncell) {  // this wavefront's rows of the tile's list
      st[j] = AT(I.b.theta, cr[j], k);
      sw[j] = AT(I.b.w, cr[j], k);
    }
  }
  diag_edge_rows(I, u, e, k, a);
  b.rue = AT(I.b.c_ru, e, k);
  b.sru = b.sth0 = b.sth1 = 0.0f;
  if (CORR) {
    b.sru = AT(I.b.s_ru, e, k);
    b.sth0 = AT(I.b.s_theta, b.c0, k);
    b.sth1 = AT(I.b.s_theta, b.c1, k);
  }
  keep(st, sw);
#pragma unroll
  for (int j = 0; j < J; ++j)
    if (w + j * HX_TILE_E < ncell) {
      s_th[(w + j * HX_TILE_E) * 64 + k] = st[j];
      s_w[(w + j * HX_TILE_E) * 64 + k] = sw[j];
    }
  __syncthreads();
#pragma unroll
  for (int sl = 0; sl < NX; ++sl) {
    b.thn[sl] = s_th[b.ac[sl] * 64 + k];
    b.wn[sl] = s_w[b.ac[sl] * 64 + k];
  }
  keep(b.thn, b.wn, b.rue, b.sru, b.sth0, b.sth1, b.fzm, b.fzp, b.dv);
  keep(a.un, a.vrow, a.pv0, a.pv1, a.pc0, a.pc1, a.ue, a.idv, a.idc);
  settle(a.wt, b.av, b.a3v);
  const EdgeDiag d = diag_edge_compute<NE, RECON>(I, e, a);
  const EdgeFlux f = tend_flux_compute<NE, CORR>(I, e, b);
  if (live) {
    store_edge_diag(I, e, k, RECON, d);
    store_edge_flux<CORR>(I, e, k, f);
  }
}

// ---------------------------------------------------------- moist coefficients
// the moist species are summed in order, their rows loaded HX_MOIST_G at a
// time before any of them is added (one round trip per batch, not per species)
constexpr int HX_MOIST_G = 8;
__device__ __forceinline__ void moist_cell(const Instance &I, int c, int k) {
  const int NM = I.n.NM;
  float t = 0.0f;
  for (int s0 = 0; s0 < NM; s0 += HX_MOIST_G) {
    float q[HX_MOIST_G];
#pragma unroll
    for (int g = 0; g < HX_MOIST_G; ++g) q[g] = s0 + g < NM ? AT(I.b.q, (s0 + g) * I.n.C + c, k) : 0.0f;
    keep(q);
#pragma unroll
    for (int g = 0; g < HX_MOIST_G; ++g)
      if (s0 + g < NM) t = t + q[g];
  }
  const float tm = up1(t);
  const float cqw = k >= 1 ? 1.0f / (1.0f + 0.5f * (t + tm)) : 1.0f;
  if (k < I.n.L) {
    AT(I.b.qtot, c, k) = t;
    AT(I.b.cqw, c, k) = cqw;
  }
}

__device__ __forceinline__ void moist_edge(const Instance &I, int e, int k) {
  const int c0 = I.m.coe[2 * e], c1 = I.m.coe[2 * e + 1];
  const int NM = I.n.NM;
  fence(c0);
  fence(c1);
  float t = 0.0f;
  for (int s0 = 0; s0 < NM; s0 += HX_MOIST_G) {
    float q0[HX_MOIST_G], q1[HX_MOIST_G];
#pragma unroll
    for (int g = 0; g < HX_MOIST_G; ++g) {
      q0[g] = s0 + g < NM ? AT(I.b.q, (s0 + g) * I.n.C + c0, k) : 0.0f;
      q1[g] = s0 + g < NM ? AT(I.b.q, (s0 + g) * I.n.C + c1, k) : 0.0f;
    }
    keep(q0, q1);
#pragma unroll
    for (int g = 0; g < HX_MOIST_G; ++g)
      if (s0 + g < NM) t = t + 0.5f * (q0[g] + q1[g]);
  }
  if (k < I.n.L) AT(I.b.cqu, e, k) = 1.0f / (1.0f + t);
}

// What opens a step, in one launch: the moist coefficients of the edges in the
// first nb0 blocks, those of the cells and (DIAG) the cells' diagnostics in the
// others; none reads what another writes.  Three launches to one: a x1.162 step
// 308 -> 302 us; x1.40962, where they took 34.3 + 15.8 + 37.3 us: 83.4.
template <int NE, bool DIAG>
KB k_begin(const Instance I, int nb0) {
  const int k = lane();
  if ((int)blockIdx.x < nb0) {
    const int e = wave_entity_first(I, nb0);
    if (e < I.n.E) moist_edge(I, e, k);
    return;
  }
  const int c = wave_entity_second(I, nb0);
  if (c >= I.n.C) return;
  if (DIAG) {
    CellVertIn<NE> a;
    cell_vert_index(I, c, a);
    cell_vert_fence(a);
    cell_vert_rows(I, I.b.u, k, a);
    keep(a.uo, a.ux, a.ia);
    settle(a.sd, a.dd, a.kt, a.rec);
    cell_vert_finish(I, c, k, a, 1);
  }
  moist_cell(I, c, k);
}

// ------------------------------------------------------ implicit coefficients
// The rows the coefficients of a column are formed from, and the coefficients
// of a level.
struct CoefIn {
  float zk, exk, thk, cqw, qt, rtpk, rbk, rtbk, exbk;
};
struct CoefOut {
  float cofwz, coftz, cofwt, a, b, cc;
};
__device__ __forceinline__ CoefIn coef_rows(const Instance &I, const float *__restrict__ exn,
                                            const float *__restrict__ theta, const float *__restrict__ rtp, int c,
                                            int k) {
  return {AT(I.z.zz, c, k),   AT(exn, c, k),  AT(theta, c, k), AT(I.b.cqw, c, k), AT(I.b.qtot, c, k),
          AT(rtp, c, k),      AT(I.z.rb, c, k), AT(I.z.rtb, c, k), AT(I.z.exb, c, k)};
}
// Level rows: fzm, fzp, rdzu, rdzw, etp, ewp of level k; neighbours by lane moves.
__device__ __forceinline__ CoefOut coef_system(const Instance &I, const CoefIn &r, int k, float fzm, float fzp,
                                               float rdzu, float rdzw, float etp, float ewp) {
  const int L = I.n.L;
  const float g = I.k.gravity, rcv = I.k.rcv, c2 = I.k.c2;
  const float zkm = up1(r.zk), exkm = up1(r.exk), thkm = up1(r.thk);
  const float rdzwm = up1(rdzw), etpm = up1(etp);
  const float ewpm = up1(ewp), ewpp = dn1(ewp);
  float cofwr = 0.0f, cofwz = 0.0f, coftz = 0.0f;
  if (k >= 1 && k < L) {
    const float iz = fzm * r.zk + fzp * zkm;
    cofwr = (0.5f * g) * iz;
    cofwz = (((c2 * iz) * rdzu) * r.cqw) * (fzm * r.exk + fzp * exkm);
    coftz = fzm * r.thk + fzp * thkm;
  }
  float cofwt = 0.0f;
  if (k < L)
    cofwt = (((((((0.5f * rcv) * r.zk) * g) * r.rbk) / (1.0f + r.qt)) * r.exk) / ((r.rtbk + r.rtpk) * r.exbk));
  const float coftz_m = up1(coftz), coftz_p = dn1(coftz), cofwt_m = up1(cofwt);
  float a = 0.0f, b = 1.0f, cc = 0.0f;
  if (k >= 1 && k < L) {
    a = (((-cofwz) * coftz_m) * rdzwm) * zkm + cofwr * rdzwm - (cofwt_m * coftz_m) * rdzwm;
    a = (a * etpm) * ewpm;
    b = (cofwz * coftz) * ((etp * rdzw) * r.zk + (etpm * rdzwm) * zkm) -
        coftz * ((etp * cofwt) * rdzw - (etpm * cofwt_m) * rdzwm) + cofwr * (etp * rdzw - etpm * rdzwm);
    b = b * ewp;
    cc = (((-cofwz) * coftz_p) * rdzw) * r.zk - cofwr * rdzw + (cofwt * coftz_p) * rdzw;
    cc = (cc * etp) * ewpp;
    if (k == L - 1) cc = 0.0f;
  }
  return {cofwz, coftz, cofwt, a, b, cc};
}
__device__ __forceinline__ void store_coefs(const Instance &I, int c, int k, float coftz, float cofwt, float cofwz,
                                            float a, float alpha, float gamma) {
  if (k > I.n.L) return;
  AT(I.b.coftz, c, k) = coftz;
  if (k < I.n.L) {
    AT(I.b.cofwz, c, k) = cofwz;
    AT(I.b.cofwt, c, k) = cofwt;
    if (I.k.store_flux) AT(I.b.atri, c, k) = a;  // export only: the acoustic column update forms a itself
    AT(I.b.alpha, c, k) = alpha;
    AT(I.b.gamma, c, k) = gamma;
  }
}

KBCOL(COLW_VC) k_vcoef(const Instance I, float dts, const float *__restrict__ exn, const float *__restrict__ theta,
              const float *__restrict__ rtp) {
  constexpr int COLW = COLW_VC;
  __shared__ float s_lev[6 * 64];
  const int w = (int)(threadIdx.x >> 6);
  const int c0 = wave_entity<COLW>();
  const bool live = c0 < I.n.C;
  const int c = live ? c0 : 0;  // every wave reaches the barriers
  const int k = lane();
  const int L = I.n.L;
  // every load first; the level k-1 and k+1 values come from neighbouring lanes
  const CoefIn r = coef_rows(I, exn, theta, rtp, c, k);
  {
    const float *const lev[6] = {I.z.fzm, I.z.fzp, I.z.rdzu, I.z.rdzw, I.z.etp, I.z.ewp};
    stage_levels<6>(s_lev, lev, w, k);
  }
  __syncthreads();
  const CoefOut o = coef_system(I, r, k, s_lev[0 * 64 + k], s_lev[1 * 64 + k], s_lev[2 * 64 + k], s_lev[3 * 64 + k],
                                s_lev[4 * 64 + k], s_lev[5 * 64 + k]);
  float a = o.a, b = o.b;
  if (coef_sweep(a, b, o.cc, k, L, dts * dts) && live) set_flag(I.b.flag);
  if (live) store_coefs(I, c, k, o.coftz, o.cofwt, o.cofwz, o.a, a, b);
}

// ------------------------------------------------------- horizontal mixing
// v8.4.1 2-D Smagorinsky mixing, once per dynamics subcycle from the
// subcycle-start state (cuda_horizontal_v841.py:205-583, host sequence
// :1270-1588; mpas_atm_dissipation_models.F smagorinsky_2d and the u/w/theta
// del2/del4 filters).  Edge density is 0.5*(rho[cell0]+rho[cell1]) of the
// current rho_zz, as the subcycle-start solve formed it.

// 2-D Smagorinsky eddy viscosity of level k (lane k) from the deformation
// sums of a cell's edge winds (smagorinsky_v841_f32)
__device__ __forceinline__ float kdiff_from_deformation(const Instance &I, int k, float dudx, float dudy, float dvdx,
                                                       float dvdy) {
  const float d11 = 2.0f * dudx, d22 = 2.0f * dvdy, d12 = dudy + dvdx;
  const float diff = d11 - d22;
  const float strain = __builtin_sqrtf(0.25f * (diff * diff) + d12 * d12);
  const float kd = fminf(I.k.strain_scale * strain, I.k.ceiling);
  // CAM floor over the top levels (native/upper_damping.rs:5-16,
  // cuda_upper_damping_v841.py:5-11): max(kdiff, base*(1 - (L-1-k)/n))
  const int L = I.n.L, ncam = I.k.cam_levels;
  if (k >= L - ncam && k < L) return fmaxf(kd, I.k.cam_base * (1.0f - (float)(L - 1 - k) / (float)ncam));
  return kd;
}




// divergence of delsq_u (laplacian_divergence_v841_f32)
template <int NE>
KB k_mix_lapdiv(const Instance I) {
  const int c = wave_entity(I);
  if (c >= I.n.C) return;
  const int k = lane();
  const int n = I.m.neoc[c];
  int e[NE];
  float x[NE], f[NE];
#pragma unroll
  for (int s = 0; s < NE; ++s) e[s] = I.m.eoc[c * NE + s];
  SlotRow<NE> fr = slot_row<NE>(I.m.mx_fdiv + c * NE);
#pragma unroll
  for (int s = 0; s < NE; ++s) fence(e[s]);
#pragma unroll
  for (int s = 0; s < NE; ++s) x[s] = AT(I.b.delsq_u, e[s], k);
  keep(x);
  settle(fr);
  slot_vals(fr, f);
  float acc = 0.0f;
#pragma unroll
  for (int s = 0; s < NE; ++s)
    if (s < n) acc = acc + f[s] * x[s];
  if (k < I.n.L) AT(I.b.delsq_div, c, k) = acc;
}

// vorticity of delsq_u (laplacian_vorticity_v841_f32)
KB k_mix_lapvort(const Instance I) {
  const int v = wave_entity(I);
  if (v >= I.n.V) return;
  const int k = lane();
  int e[3];
  float x[3], f[3];
#pragma unroll
  for (int s = 0; s < 3; ++s) e[s] = I.m.eov[3 * v + s];
  SlotRow<3> fr = slot_row<3>(I.m.mx_fvort + 3 * v);
#pragma unroll
  for (int s = 0; s < 3; ++s) fence(e[s]);
#pragma unroll
  for (int s = 0; s < 3; ++s) x[s] = AT(I.b.delsq_u, e[s], k);
  keep(x);
  settle(fr);
  slot_vals(fr, f);
  float acc = 0.0f;
#pragma unroll
  for (int s = 0; s < 3; ++s) acc = acc + f[s] * x[s];
  if (k < I.n.L) AT(I.b.delsq_vort, v, k) = acc;
}

// del2 of theta and of w (theta_filter_lap2_v841_f32, w_filter_lap2_v841_f32).
// Without the fourth-order part (MIX4 false) the results go straight to the
// Euler pools.  LAP: also the divergence and, at the vertices the cell owns,
// the vorticity of delsq_u, from the cell's own and outward edges as in
// k_diag_cv; every weight of a slot comes in one record row, where a row each
// and a scalar load per edge cost the wavefront their issue.  The three passes
// took 30.5 + 13.4 + 16.7 us at x1.40962, this one 47.0 (126 MB counted once,
// 2.7 TB/s: bound by the issue of its 41 row loads).
template <int NE, bool MIX4, bool LAP>
KB k_mix_cell(const Instance I) {
  const int c = wave_entity(I);
  if (c >= I.n.C) return;
  const int k = lane();
  const int L = I.n.L;
  const int n = I.m.neoc[c];
  const int code = LAP ? I.m.vcode[c] : 0;
  int e[NE], x[NE], o[NE], vo[NE];
#pragma unroll
  for (int s = 0; s < NE; ++s) {
    vo[s] = LAP ? I.m.voc[c * NE + s] : 0;
    e[s] = LAP ? I.m.eoc[c * NE + s] : 0;
    x[s] = LAP ? I.m.vx[c * NE + s] : 0;
    o[s] = I.m.ocell[c * NE + s];
  }
  SlotRow<HX_ROW> rec = slot_row<HX_ROW>(I.m.mx_rec + c * HX_ROW);
  const float thc = AT(I.b.theta, c, k), rhc = AT(I.b.c_rho, c, k), wc = AT(I.b.w, c, k);
  const float kdc = AT(I.b.kdiff, c, k);
  const float erw = MIX4 ? 0.0f : AT(I.b.euler_rw, c, k);
  fence(code);
#pragma unroll
  for (int s = 0; s < NE; ++s) {
    fence(e[s]);
    fence(x[s]);
    fence(o[s]);
    fence(vo[s]);
  }
  float tho[NE], rho[NE], wo[NE], kdo[NE], uo[NE], ux[NE];
#pragma unroll
  for (int s = 0; s < NE; ++s) {
    tho[s] = AT(I.b.theta, o[s], k);
    rho[s] = AT(I.b.c_rho, o[s], k);
    wo[s] = AT(I.b.w, o[s], k);
    kdo[s] = AT(I.b.kdiff, o[s], k);
    uo[s] = LAP ? AT(I.b.delsq_u, e[s], k) : 0.0f;
    ux[s] = LAP ? AT(I.b.delsq_u, x[s], k) : 0.0f;
  }
  keep(tho, rho, wo, kdo);
  if (LAP) keep(uo, ux);
  settle(rec);
  if (LAP) {
    float acc = 0.0f;
    float uq = uo[2];  // the edge row of slot s - 1: of the last slot for s = 0
#pragma unroll
    for (int s = 3; s < NE; ++s) uq = s < n ? uo[s] : uq;
#pragma unroll
    for (int s = 0; s < NE; ++s)
      if (s < n) {
        const float up = uo[s];
        const int r = s * HX_VREC;
        acc = acc + rec[r + 3] * up;
        if (code >> (16 + s) & 1) {
          const int last = code >> (2 * s) & 3;
          const float u0 = last == 0 ? uq : up, u1 = last == 2 ? uq : ux[s],
                      u2 = last == 2 ? ux[s] : last == 1 ? uq : up;
          float z = 0.0f + rec[r] * u0;
          z = z + rec[r + 1] * u1;
          z = z + rec[r + 2] * u2;
          if (k < L) AT(I.b.delsq_vort, vo[s], k) = z;
        }
        uq = up;
      }
    if (k < L) AT(I.b.delsq_div, c, k) = acc;
  }
  float lap = 0.0f, tend = 0.0f, lapw = 0.0f, tendw = 0.0f;
#pragma unroll
  for (int s = 0; s < NE; ++s) {
    // cell0/cell1 of edge s in cellsOnEdge order
    const int r = s * HX_VREC;
    const float f2 = rec[r + 4], fw = rec[r + 5], d2 = rec[r + 6];
    const bool first = rec[r + 7] > 0.0f;
    const float th0 = first ? thc : tho[s], th1 = first ? tho[s] : thc;
    const float r0 = first ? rhc : rho[s], r1 = first ? rho[s] : rhc;
    const float w0 = first ? wc : wo[s], w1 = first ? wo[s] : wc;
    const float k0 = first ? kdc : kdo[s], k1 = first ? kdo[s] : kdc;
    const float rho_e = 0.5f * (r0 + r1);
    const float rho_em = up1(rho_e);
    const float k0m = up1(k0), k1m = up1(k1);
    if (s < n) {
      const float flux = (f2 * (th1 - th0)) * rho_e;
      lap = lap + flux;
      tend = tend + ((flux * 0.5f) * (k0 + k1)) * d2;
      const float fluxw = (fw * (rho_e + rho_em)) * (w1 - w0);
      lapw = lapw + fluxw;
      const float sum_k = ((k0 + k1) + k0m) + k1m;
      tendw = tendw + ((fluxw * d2) * 0.25f) * sum_k;
    }
  }
  if (k == 0 || k >= L) {
    lapw = 0.0f;
    tendw = 0.0f;
  }
  if (k < L) {
    AT(I.b.delsq_theta, c, k) = lap;
    AT(I.b.euler_theta, c, k) = tend;
    AT(I.b.delsq_w, c, k) = lapw;
  }
  if (MIX4) {
    if (k <= L) AT(I.b.mix_tw, c, k) = tendw;
  } else if (k <= L) {
    AT(I.b.euler_rw, c, k) = erw + tendw;
  }
}

// del4 of theta and of w (theta_filter_lap4_v841_f32, w_filter_lap4_v841_f32), then the w pool
template <int NE>
__device__ __forceinline__ void mix_cell4(const Instance &I, int c, int k) {
  const int L = I.n.L;
  const int n = I.m.neoc[c];
  int o[NE];
#pragma unroll
  for (int s = 0; s < NE; ++s) o[s] = I.m.ocell[c * NE + s];
  SlotRow<NE> sgr = slot_row<NE>(I.m.csign + c * NE), f4r = slot_row<NE>(I.m.mx_f4 + c * NE);
  const float dtc = AT(I.b.delsq_theta, c, k), dwc = AT(I.b.delsq_w, c, k);
  float tend = AT(I.b.euler_theta, c, k);
  float tendw = AT(I.b.mix_tw, c, k);
  const float erw = AT(I.b.euler_rw, c, k);
#pragma unroll
  for (int s = 0; s < NE; ++s) fence(o[s]);
  float dto[NE], dwo[NE];
#pragma unroll
  for (int s = 0; s < NE; ++s) {
    dto[s] = AT(I.b.delsq_theta, o[s], k);
    dwo[s] = AT(I.b.delsq_w, o[s], k);
  }
  keep(dto, dwo);
  settle(sgr, f4r);
  float sg[NE], f4[NE];
  slot_vals(sgr, sg);
  slot_vals(f4r, f4);
  const bool wlev = k >= 1 && k < L;
#pragma unroll
  for (int s = 0; s < NE; ++s)
    if (s < n) {
      const bool first = sg[s] > 0.0f;
      const float t0 = first ? dtc : dto[s], t1 = first ? dto[s] : dtc;
      const float w0 = first ? dwc : dwo[s], w1 = first ? dwo[s] : dwc;
      tend = tend - f4[s] * (t1 - t0);
      if (wlev) tendw = tendw - f4[s] * (w1 - w0);
    }
  if (k < L) AT(I.b.euler_theta, c, k) = tend;
  if (k <= L) AT(I.b.euler_rw, c, k) = erw + tendw;
}

// del4 of u (momentum_filter_lap4_v841_f32): pool - rho_e*((ddiv*r_dc) - (dvort*r_dv))
__device__ __forceinline__ void mix_edge4(const Instance &I, int e, int k) {
  const int c0 = I.m.coe[2 * e], c1 = I.m.coe[2 * e + 1];
  const int v0 = I.m.voe[2 * e], v1 = I.m.voe[2 * e + 1];
  const float d0 = AT(I.b.delsq_div, c0, k), d1 = AT(I.b.delsq_div, c1, k);
  const float z0 = AT(I.b.delsq_vort, v0, k), z1 = AT(I.b.delsq_vort, v1, k);
  const float r0 = AT(I.b.c_rho, c0, k), r1 = AT(I.b.c_rho, c1, k);
  const float eru = AT(I.b.euler_ru, e, k);
  const float rdc = uni_load(I.m.mx_rdc + e), rdv = uni_load(I.m.mx_rdv + e);
  const float rho_e = 0.5f * (r0 + r1);
  const float diffusion = rho_e * ((d1 - d0) * rdc - (z1 - z0) * rdv);
  if (k < I.n.L) AT(I.b.euler_ru, e, k) = eru - diffusion;
}

// the fourth-order part, after k_mix_cell: edges of the momentum pool in the
// first nb0 blocks, cells of the theta and w pools in the others: 29.9 +
// 18.1 us as two launches at x1.40962, 47.4 as one; on small meshes the launch
// (4 to 5 us) is most of either.
template <int NE>
KB k_mix4(const Instance I, int nb0) {
  const int k = lane();
  if ((int)blockIdx.x < nb0) {
    const int e = wave_entity_first(I, nb0);
    if (e < I.n.E) mix_edge4(I, e, k);
  } else {
    const int c = wave_entity_second(I, nb0);
    if (c < I.n.C) mix_cell4<NE>(I, c, k);
  }
}

// ------------------------------------------------------------ subcycle start
// MIX: also the 2-D Smagorinsky kdiff of the cell (mix_kdiff_value's
// arithmetic); MOIST: moisture species present
template <int NE, bool MIX, bool MOIST>
KB k_sub_cell(const Instance I) {
  const int c = wave_entity(I);
  if (c >= I.n.C) return;
  const int k = lane();
  const int L = I.n.L;
  const int n = I.m.neoc[c];
  int e[NE];
#pragma unroll
  for (int s = 0; s < NE; ++s) e[s] = I.m.eoc[c * NE + s];
  SlotRow<NE> sd = slot_row<NE>(I.m.csdv + c * NE);
  SlotRow<NE> c2 = {0.0f}, s2 = {0.0f}, cs = {0.0f};
  if (MIX) {
    c2 = slot_row<NE>(I.m.defc2 + c * NE);
    s2 = slot_row<NE>(I.m.defs2 + c * NE);
    cs = slot_row<NE>(I.m.defcs + c * NE);
  }
  const float ia = uni_load(I.m.invarea + c);
  const float rdzw = AT(I.z.rdzw, 0, k), rdzu = AT(I.z.rdzu, 0, k);
  const float fzm = AT(I.z.fzm, 0, k), fzp = AT(I.z.fzp, 0, k);
  const float rho_p = AT(I.b.s_rho_p, c, k);
  const float qt = MOIST ? AT(I.b.qtot, c, k) : 0.0f;
  const float rb = MOIST ? AT(I.z.rb, c, k) : 0.0f;
  const float cqw = MOIST ? AT(I.b.cqw, c, k) : 0.0f;
  const float rw_k = AT(I.b.c_rw, c, k);
  const float pp_k = AT(I.b.pp, c, k);
#pragma unroll
  for (int s = 0; s < NE; ++s) fence(e[s]);
  float xv[NE], un[NE], vn[NE];
#pragma unroll
  for (int s = 0; s < NE; ++s) {
    xv[s] = AT(I.b.c_ru, e[s], k);
    un[s] = MIX ? AT(I.b.u, e[s], k) : 0.0f;
    vn[s] = MIX ? AT(I.b.v, e[s], k) : 0.0f;
  }
  const float prho = I.k.physics ? AT(I.b.phys_rho, c, k) : 0.0f;  // the buffer exists with physics only
  keep(xv);
  if (MIX) keep(un, vn);
  settle(sd, c2, s2, cs);
  float kd = 0.0f;
  if (MIX) {
    float dudx = 0.0f, dudy = 0.0f, dvdx = 0.0f, dvdy = 0.0f;
#pragma unroll
    for (int s = 0; s < NE; ++s)
      if (s < n) {
        dudx = (dudx + c2[s] * un[s]) - cs[s] * vn[s];
        dudy = (dudy + cs[s] * un[s]) - s2[s] * vn[s];
        dvdx = (dvdx + cs[s] * un[s]) + c2[s] * vn[s];
        dvdy = (dvdy + s2[s] * un[s]) + cs[s] * vn[s];
      }
    kd = kdiff_from_deformation(I, k, dudx, dudy, dvdx, dvdy);
  }
  float acc = 0.0f;
#pragma unroll
  for (int s = 0; s < NE; ++s)
    if (s < n) acc = acc + sd[s] * xv[s];
  acc = acc * ia;
  const float g = I.k.gravity;
  const float dpdz = MOIST ? (-g) * (rb * qt + rho_p * (1.0f + qt)) : (-g) * rho_p;
  // 0 - x, not -x: a zero divergence gives +0 (density_tendency_f32)
  const float trho = (0.0f - acc) - rdzw * (dn1(rw_k) - rw_k);
  const float pp_m1 = up1(pp_k);
  const float dpdzm = up1(dpdz);
  float erw = 0.0f;
  if (k >= 1 && k < L) {
    const float inner = rdzu * (pp_k - pp_m1) - (fzm * dpdz + fzp * dpdzm);
    erw = MOIST ? 0.0f - cqw * inner : 0.0f - inner;  // euler_w(_moist_v841)_f32
  }
  if (k < L) {
    const float tr = I.k.physics ? trho + prho : trho;
    AT(I.b.dpdz, c, k) = dpdz;
    AT(I.b.tend_rho, c, k) = tr;
    AT(I.b.hdiv, c, k) = acc;  // stage-1 mass-flux divergence of the current ru
    if (MIX) AT(I.b.kdiff, c, k) = kd;
  }
  if (k <= L) AT(I.b.euler_rw, c, k) = erw;
}

// MIX: also add the del2 u increment of the 2-D Smagorinsky mixing to the
// pool (mixing.py del2 u term, in the same pass; kdiff is final by then)
template <bool MIX>
KB k_sub_edge(const Instance I) {
  const int e = wave_entity(I);
  if (e >= I.n.E) return;
  const int k = lane();
  const int c0 = I.m.coe[2 * e], c1 = I.m.coe[2 * e + 1];
  int v0 = 0, v1 = 0;
  if (MIX) {
    v0 = I.m.voe[2 * e];
    v1 = I.m.voe[2 * e + 1];
  }
  fence(c0);
  fence(c1);
  fence(v0);
  fence(v1);
  // every row first: the pool's, then (with mixing) del2 u's: divergence,
  // vorticity, kdiff and rho of the edge's cells and vertices
  const float *pp = I.b.pp, *zz = I.z.zz, *dz = I.b.dpdz;
  const float idc = uni_load(I.m.invdc + e);
  const float pp0 = AT(pp, c0, k), pp1 = AT(pp, c1, k), zz0 = AT(zz, c0, k), zz1 = AT(zz, c1, k);
  const float dz0 = AT(dz, c0, k), dz1 = AT(dz, c1, k), zxu = AT(I.z.zxu, e, k), cqu = AT(I.b.cqu, e, k);
  float d0 = 0.0f, d1 = 0.0f, z0 = 0.0f, z1 = 0.0f, kd0 = 0.0f, kd1 = 0.0f, r0 = 0.0f, r1 = 0.0f;
  float midc = 0.0f, midv = 0.0f, del2 = 0.0f;
  if (MIX) {
    d0 = AT(I.b.divergence, c0, k);
    d1 = AT(I.b.divergence, c1, k);
    z0 = AT(I.b.vorticity, v0, k);
    z1 = AT(I.b.vorticity, v1, k);
    kd0 = AT(I.b.kdiff, c0, k);
    kd1 = AT(I.b.kdiff, c1, k);
    r0 = AT(I.b.c_rho, c0, k);
    r1 = AT(I.b.c_rho, c1, k);
    midc = uni_load(I.m.mx_idc + e);
    midv = uni_load(I.m.mx_idv + e);
    del2 = uni_load(I.m.mx_del2 + e);
  }
  keep(pp0, pp1, zz0, zz1, dz0, dz1, zxu, cqu);
  if (MIX) keep(d0, d1, z0, z1, kd0, kd1, r0, r1);
  const float a = ((pp1 - pp0) * idc) / (0.5f * (zz1 + zz0));
  const float bb = (0.5f * zxu) * (dz0 + dz1);
  const float pool = (0.0f - cqu) * (a - bb);
  if (MIX) {
    // del2 u at level k: the increment added to the u pool, and delsq_u
    const float lap = (d1 - d0) * midc - (z1 - z0) * midv;
    const float kedge = 0.5f * (kd0 + kd1);
    const float rho_e = 0.5f * (r0 + r1);
    const float inc = ((rho_e * kedge) * lap) * del2;
    if (k < I.n.L) {
      if (I.k.mix4) AT(I.b.delsq_u, e, k) = lap;
      AT(I.b.euler_ru, e, k) = pool + inc;
    }
  } else {
    if (k < I.n.L) AT(I.b.euler_ru, e, k) = pool;
  }
}

// ---------------------------------------------------------- stage tendencies

// momentum tendency of one stage (dynamics.py:223-268, dynamics_v841.py:128-185);
// returns lane k's tend_ru value, stored for levels k < L.
// REFW: a reference wind is set, whose Coriolis force is taken out again.
// With u_init and v_init zero (and finite weights, angles and f, checked at
// create) every term of that sum is a signed zero, and the sum it is
// subtracted from started at +0 and so is never -0: leaving the terms out
// keeps the bits.  Without the terms a wavefront issues 182 vector
// instructions and 40 loads instead of 274 and 45; a launch takes 64.7 us
// instead of 68.8 (x1.40962), what is left is the row loads' own rate.
template <int NE, bool REFW>
__device__ __forceinline__ float tend_mom_edge(const Instance &I, int e, int k) {
  constexpr int NX = 2 * NE - 2;
  const int L = I.n.L;
  const int c0 = I.m.coe[2 * e], c1 = I.m.coe[2 * e + 1];
  int nb[NX];
#pragma unroll
  for (int s = 0; s < NX; ++s) nb[s] = I.m.eoe[e * NX + s];
  const int nn = I.m.neoe[e];
  SlotRow<NX> wt = slot_row<NX>(I.m.woe + e * NX), ca = {0.0f}, sa = {0.0f};
  float fe = 0.0f, ui = 0.0f, vi = 0.0f;
  if (REFW) {
    ca = slot_row<NX>(I.m.ecos + e * NX);
    sa = slot_row<NX>(I.m.esin + e * NX);
    fe = uni_load(I.m.fedge + e);
    ui = AT(I.z.uinit, 0, k);
    vi = AT(I.z.vinit, 0, k);
  }
  const float idc = uni_load(I.m.invdc + e);
  const float fzm = AT(I.z.fzm, 0, k), fzp = AT(I.z.fzp, 0, k), rdzw = AT(I.z.rdzw, 0, k);
  const float u_k = AT(I.b.u, e, k);
  const float rw0 = AT(I.b.c_rw, c0, k), rw1 = AT(I.b.c_rw, c1, k);
  const float pve = AT(I.b.pv_edge, e, k);
  float un[NX], pvn[NX];
#pragma unroll
  for (int s = 0; s < NX; ++s) {
    un[s] = AT(I.b.u, nb[s], k);
    pvn[s] = AT(I.b.pv_edge, nb[s], k);
  }
  const float rho0 = AT(I.b.c_rho, c0, k), rho1 = AT(I.b.c_rho, c1, k);
  const float ke0 = AT(I.b.ke, c0, k), ke1 = AT(I.b.ke, c1, k);
  const float hd0 = AT(I.b.hdiv, c0, k), hd1 = AT(I.b.hdiv, c1, k);
  const float eru = AT(I.b.euler_ru, e, k);
  const float pru = I.k.physics ? AT(I.b.phys_ru, e, k) : 0.0f;  // the buffer exists with physics only
  keep(un, pvn);
  keep(u_k, rw0, rw1, pve, rho0, rho1, ke0, ke1, hd0, hd1, eru, idc);
  settle(wt);
  if (REFW) {
    keep(fe);
    settle(ca, sa);
  }
  const float u_m1 = up1(u_k), u_m2 = up1(up1(u_k)), u_p1 = dn1(u_k);
  const float rwe = 0.5f * (rw0 + rw1);
  float wduz = 0.0f;
  if (k == 1 || k == L - 1) {
    wduz = rwe * (fzm * u_k + fzp * u_m1);
  } else if (k >= 2 && k < L - 1) {
    wduz = flux3(u_m2, u_m1, u_k, u_p1, rwe, 1.0f);
  }
  const float wduz_p = dn1(wduz);
  const float initial = (-rdzw) * (wduz_p - wduz);
  float qq = 0.0f;
#pragma unroll
  for (int s = 0; s < NX; ++s)
    if (s < nn) {
      const float work_pv = 0.5f * (pve + pvn[s]);
      qq = qq + (wt[s] * un[s]) * work_pv;
    }
  if (REFW) {
#pragma unroll
    for (int s = 0; s < NX; ++s)
      if (s < nn) {
        const float ref_u = ui * ca[s] - vi * sa[s];
        qq = qq - (wt[s] * ref_u) * fe;
      }
  }
  const float rho_edge = 0.5f * (rho0 + rho1);
  const float horiz = rho_edge * (qq - (ke1 - ke0) * idc);
  float t = (initial + horiz) - (u_k * 0.5f) * (hd0 + hd1);
  // upper-level Rayleigh damping of u, before the Euler pool is added
  // (native/upper_damping.rs:18-31; cuda_upper_damping_v841.py:12-18)
  const int nray = I.k.ray_levels;
  if (k >= L - nray && k < L) t = t - (rho_edge * u_k) * ((float)(k - (L - nray) + 1) * I.k.ray_inverse);
  const float tr = I.k.physics ? (t + eru) + pru : t + eru;
  if (k < L) AT(I.b.tend_ru, e, k) = tr;
  return tr;
}

template <int NE, bool REFW>
KB k_tend_mom(const Instance I) {
  const int e = wave_entity(I);
  if (e >= I.n.E) return;
  tend_mom_edge<NE, REFW>(I, e, lane());
}

// the momentum tendency and the first acoustic substep's edge update
// (ru_p = dts * tend_ru, acoustic_v841.py:296-330) in one pass.  The running
// sum ru_avg equals ru_p after one substep; it is stored only when a later
// substep reads it back (with two substeps the second forms p1 + p2 from
// ru_p, with one the recovery reads ru_p itself).  ru_p itself is stored
// only for a second substep's edge update or, at stage 3, for the step's
// output: the first substep's column update and a one-substep stage's
// recovery form dts * tend_ru from tend_ru.
template <int NE, bool REFW>
KB k_tend_mom_ac(const Instance I, float dts, int store_avg, int store_rup) {
  const int e = wave_entity(I);
  if (e >= I.n.E) return;
  const int k = lane();
  const float tr = tend_mom_edge<NE, REFW>(I, e, k);
  if (k < I.n.L) {
    const float p = dts * tr;
    if (store_rup) AT(I.b.ru_p, e, k) = p;
    if (store_avg) AT(I.b.ru_avg, e, k) = p;
  }
}

// theta and w edge fluxes of edge e with the 3rd-order upwind-blended
// stencil (driver.py:1003-1034, 1140-1170) and, at stages 2-3, the theta RK
// correction flux (cuda_dynamics_v841.py:209-247)
// CORR: stages 2 and 3, which add the theta RK correction flux
template <int NE>
struct EdgeFluxIn {
  float thn[2 * NE - 2], wn[2 * NE - 2];
  SlotRow<2 * NE - 2> av, a3v;
  float rue, sru, sth0, sth1, fzm, fzp, dv;
  int na;
  int c0, c1, ac[2 * NE - 2];  // scalar index loads
};
template <int NE, bool CORR>
__device__ __forceinline__ void tend_flux_index(const Instance &I, int e, int k, EdgeFluxIn<NE> &b) {
  constexpr int NX = 2 * NE - 2;
  b.c0 = I.m.coe[2 * e];
  b.c1 = I.m.coe[2 * e + 1];
#pragma unroll
  for (int s = 0; s < NX; ++s) b.ac[s] = I.m.advc[e * NX + s];
  b.na = I.m.nadv[e];
  b.av = slot_row<NX>(I.m.adv + e * NX);
  b.a3v = slot_row<NX>(I.m.adv3 + e * NX);
  b.dv = CORR ? uni_load(I.m.dv + e) : 0.0f;
  b.fzm = AT(I.z.fzm, 0, k);
  b.fzp = AT(I.z.fzp, 0, k);
}
template <int NE>
__device__ __forceinline__ void tend_flux_fence(const EdgeFluxIn<NE> &b) {
  fence(b.c0);
  fence(b.c1);
#pragma unroll
  for (int s = 0; s < 2 * NE - 2; ++s) fence(b.ac[s]);
}
template <int NE, bool CORR>
__device__ __forceinline__ void tend_flux_rows(const Instance &I, int e, int k, EdgeFluxIn<NE> &b) {
  constexpr int NX = 2 * NE - 2;
#pragma unroll
  for (int s = 0; s < NX; ++s) {
    b.thn[s] = AT(I.b.theta, b.ac[s], k);
    b.wn[s] = AT(I.b.w, b.ac[s], k);
  }
  b.rue = AT(I.b.c_ru, e, k);
  b.sru = b.sth0 = b.sth1 = 0.0f;
  if (CORR) {
    b.sru = AT(I.b.s_ru, e, k);
    b.sth0 = AT(I.b.s_theta, b.c0, k);
    b.sth1 = AT(I.b.s_theta, b.c1, k);
  }
}
template <int NE, bool CORR>
__device__ __forceinline__ EdgeFluxIn<NE> tend_flux_load(const Instance &I, int e, int k) {
  EdgeFluxIn<NE> b;
  tend_flux_index<NE, CORR>(I, e, k, b);
  tend_flux_fence(b);
  tend_flux_rows<NE, CORR>(I, e, k, b);
  settle(b.av, b.a3v);
  return b;
}
template <int NE, bool CORR>
__device__ __forceinline__ EdgeFlux tend_flux_compute(const Instance &I, int e, const EdgeFluxIn<NE> &b) {
  constexpr int NX = 2 * NE - 2;
  const float rue_m = up1(b.rue);
  const float coef = I.k.coef3;
  const float rui = b.fzm * b.rue + b.fzp * rue_m;
  const float sv_t = cs1(b.rue), sv_w = cs1(rui);
  float et = 0.0f, ew = 0.0f;
#pragma unroll
  for (int s = 0; s < NX; ++s)
    if (s < b.na) {
      const float a = b.av[s], a3 = b.a3v[s];
      et = et + (a + (coef * sv_t) * a3) * b.thn[s];
      ew = ew + (a + (coef * sv_w) * a3) * b.wn[s];
    }
  EdgeFlux f;
  f.th = b.rue * et;
  f.corr = CORR ? ((b.dv * (b.sru - b.rue)) * 0.5f) * (b.sth1 + b.sth0) : 0.0f;
  f.w = rui * ew;
  return f;
}
template <int NE, bool CORR>
__device__ __forceinline__ EdgeFlux tend_flux_values(const Instance &I, int e, int k) {
  return tend_flux_compute<NE, CORR>(I, e, tend_flux_load<NE, CORR>(I, e, k));
}
template <bool CORR>
__device__ __forceinline__ void store_edge_flux(const Instance &I, int e, int k, EdgeFlux f) {
  if (k < I.n.L) {
    AT(I.b.fth, e, k) = f.th;
    if (CORR) AT(I.b.fcorr, e, k) = f.corr;
    if (k >= 1) AT(I.b.fw, e, k) = f.w;
  }
}

template <int NE, bool CORR>
KB k_tend_flux(const Instance I) {
  const int e = wave_entity(I);
  if (e >= I.n.E) return;
  const int k = lane();
  store_edge_flux<CORR>(I, e, k, tend_flux_values<NE, CORR>(I, e, k));
}

// Theta and w tendencies of one stage in a cell's column.  CORR: stages 2 and
// 3 (the theta RK correction flux); MIX: horizontal mixing on (its theta
// increment is added).  The column rows are read once; vertical neighbours by
// shuffles.
template <int NE>
struct ThetaIn {
  float th, ths, rwc, rws, eth, prt;
  float fth[NE], fco[NE];
};
template <int NE>
struct WIn {
  float ww, zz, erw;
  float fwv[NE], tru[NE], zb[NE], zb3[NE];
};
template <int NE, bool CORR, bool MIX>
__device__ __forceinline__ void theta_rows(const Instance &I, const int (&e)[NE], int c, int k, ThetaIn<NE> &t) {
  t.th = AT(I.b.theta, c, k);
  t.ths = AT(I.b.s_theta, c, k);
  t.rwc = AT(I.b.c_rw, c, k);
  t.rws = AT(I.b.s_rw, c, k);
  t.eth = MIX ? AT(I.b.euler_theta, c, k) : 0.0f;
#pragma unroll
  for (int s = 0; s < NE; ++s) {
    t.fth[s] = AT(I.b.fth, e[s], k);
    t.fco[s] = CORR ? AT(I.b.fcorr, e[s], k) : 0.0f;
  }
  t.prt = I.k.physics ? AT(I.b.phys_rt, c, k) : 0.0f;  // the buffer exists with physics only
}
template <int NE>
__device__ __forceinline__ void w_rows(const Instance &I, const int (&e)[NE], int c, int k, WIn<NE> &t) {
  t.ww = AT(I.b.w, c, k);
  t.zz = AT(I.z.zz, c, k);
  t.erw = AT(I.b.euler_rw, c, k);
#pragma unroll
  for (int s = 0; s < NE; ++s) {
    t.fwv[s] = AT(I.b.fw, e[s], k);
    t.tru[s] = AT(I.b.tend_ru, e[s], k);
    t.zb[s] = AT(I.z.zb, c * NE + s, k);
    t.zb3[s] = AT(I.z.zb3, c * NE + s, k);
  }
}
template <int NE, bool CORR, bool MIX>
__device__ __forceinline__ float theta_tendency(const Instance &I, const ThetaIn<NE> &t, const float (&sg)[NE],
                                                float ia, int n, int k, float fzm, float fzp, float rdzw) {
  const int L = I.n.L;
  const float coef = I.k.coef3;
  const float th_m1 = up1(t.th), th_m2 = up1(th_m1), th_p1 = dn1(t.th), ths_m1 = up1(t.ths);
  float vf = 0.0f;
  if (k == 1) {
    vf = t.rwc * (fzm * t.th + fzp * th_m1);
    vf = vf + (t.rws - t.rwc) * (fzm * t.ths + fzp * ths_m1);
  } else if (k >= 2 && k < L - 1) {
    vf = flux3(th_m2, th_m1, t.th, th_p1, t.rwc, coef);
    vf = vf + (t.rws - t.rwc) * (fzm * t.ths + fzp * ths_m1);
  } else if (k == L - 1) {
    vf = t.rws * (fzm * t.th + fzp * th_m1);
  }
  const float vf_p = dn1(vf);
  float r = 0.0f;
#pragma unroll
  for (int s = 0; s < NE; ++s)
    if (s < n) r = r - sg[s] * t.fth[s];
  if (CORR) {
#pragma unroll
    for (int s = 0; s < NE; ++s)
      if (s < n) r = r - sg[s] * t.fco[s];
  }
  r = r * ia;
  const float trt = r - rdzw * (vf_p - vf);
  const float tmix = MIX ? trt + t.eth : trt;
  return I.k.physics ? tmix + t.prt : tmix;
}
template <int NE>
__device__ __forceinline__ float w_tendency(const Instance &I, const WIn<NE> &t, float rwc, const float (&sg)[NE],
                                            float ia, int n, int k, float fzm, float fzp, float rdzu) {
  const int L = I.n.L;
  const float rwc_m1 = up1(rwc);
  const float ww_m1 = up1(t.ww), ww_m2 = up1(ww_m1), ww_p1 = dn1(t.ww), zz_m1 = up1(t.zz);
  float wf = 0.0f;
  if (k == 1 || k == L - 1) {
    wf = (0.25f * (rwc + rwc_m1)) * (t.ww + ww_m1);
  } else if (k >= 2 && k < L - 1) {
    wf = flux3(ww_m2, ww_m1, t.ww, ww_p1, 0.5f * (rwc + rwc_m1), 1.0f);
  }
  const float wf_p = dn1(wf);
  float q = 0.0f;
#pragma unroll
  for (int s = 0; s < NE; ++s)
    if (s < n) q = q - sg[s] * t.fwv[s];
  q = q * ia;
  q = q - rdzu * (wf_p - wf);
  q = q + t.erw;
#pragma unroll
  for (int s = 0; s < NE; ++s)
    if (s < n) {
      const float tk = t.tru[s];
      const float flux = sg[s] * (fzm * tk + fzp * up1(tk));
      q = q - (t.zb[s] + cs1(tk) * t.zb3[s]) * flux;
    }
  return k >= 1 && k < L ? q * (fzm * t.zz + fzp * zz_m1) : 0.0f;
}
__device__ __forceinline__ void store_tend(const Instance &I, int c, int k, float rt, float rw) {
  if (k < I.n.L) AT(I.b.tend_rt, c, k) = rt;
  if (k <= I.n.L) AT(I.b.tend_rw, c, k) = rw;
}

template <int NE, bool CORR, bool MIX>
KB k_tend_cell(const Instance I) {
  const int c = wave_entity(I);
  if (c >= I.n.C) return;
  const int k = lane();
  const int n = I.m.neoc[c];
  int e[NE];
#pragma unroll
  for (int s = 0; s < NE; ++s) e[s] = I.m.eoc[c * NE + s];
  SlotRow<NE> sgr = slot_row<NE>(I.m.csign + c * NE);
  const float ia = uni_load(I.m.invarea + c);
  const float fzm = AT(I.z.fzm, 0, k), fzp = AT(I.z.fzp, 0, k);
  const float rdzw = AT(I.z.rdzw, 0, k), rdzu = AT(I.z.rdzu, 0, k);
#pragma unroll
  for (int s = 0; s < NE; ++s) fence(e[s]);
  ThetaIn<NE> t;
  WIn<NE> v;
  theta_rows<NE, CORR, MIX>(I, e, c, k, t);
  w_rows<NE>(I, e, c, k, v);
  keep(t.fth, v.fwv, v.tru, v.zb, v.zb3);
  if (CORR) keep(t.fco);
  settle(sgr);
  float sg[NE];
  slot_vals(sgr, sg);
  const float rt = theta_tendency<NE, CORR, MIX>(I, t, sg, ia, n, k, fzm, fzp, rdzw);
  store_tend(I, c, k, rt, w_tendency<NE>(I, v, t.rwc, sg, ia, n, k, fzm, fzp, rdzu));
}

// ----------------------------------------------------------- acoustic substep
// ru_p + divergence-damping increment of edge e at level k (mixing.py:851-945)
// OLD0: the damped substep was a stage's first, whose rtheta_pp_old is zero
// (then neither stored nor read; x - 0 keeps the bits of x)
template <bool OLD0 = false>
__device__ __forceinline__ float damped_ru_p(const Instance &I, int e, int k, float rp, float coefficient) {
  const int c0 = I.m.coe[2 * e], c1 = I.m.coe[2 * e + 1];
  const float d0 = AT(I.b.rtheta_pp, c0, k) - (OLD0 ? 0.0f : AT(I.b.rtheta_pp_old, c0, k));
  const float d1 = AT(I.b.rtheta_pp, c1, k) - (OLD0 ? 0.0f : AT(I.b.rtheta_pp_old, c1, k));
  const float den = AT(I.b.s_theta, c0, k) + AT(I.b.s_theta, c1, k);
  return rp + ((coefficient * (d0 - d1)) * (1.0f - 0.0f)) / den;
}

// FIRST: the first substep (ru_p = dts * tend_ru).  DAMP: apply the previous
// substep's divergence damping to ru_p first (the same update k_divdamp
// makes, fused into this pass over the edges).  AVGRP: this is the second of
// two substeps and ru_avg was not stored at the first, where it equals the
// undamped ru_p read here (p1 + p2, the same operands in the same order as
// ru_avg + p).  Loads first, stores last.
template <bool FIRST, bool DAMP, bool AVGRP>
KB k_ac_edge(const Instance I, float dts, float damp_coef) {
  const int e = wave_entity(I);
  if (e >= I.n.E) return;
  const int k = lane();
  if (k >= I.n.L) return;
  if (FIRST) {
    const float p = dts * AT(I.b.tend_ru, e, k);
    AT(I.b.ru_p, e, k) = p;
    AT(I.b.ru_avg, e, k) = p;
    return;
  }
  const int c0 = I.m.coe[2 * e], c1 = I.m.coe[2 * e + 1];
  const float idc = uni_load(I.m.invdc + e);
  const float tr = AT(I.b.tend_ru, e, k);
  const float rp_raw = AT(I.b.ru_p, e, k);
  const float ra_in = AVGRP ? 0.0f : AT(I.b.ru_avg, e, k);
  const float cqu = AT(I.b.cqu, e, k), zxu = AT(I.z.zxu, e, k);
  fence(c0);
  fence(c1);
  const float tp0 = AT(I.b.rtheta_pp, c0, k), tp1 = AT(I.b.rtheta_pp, c1, k);
  const float z0 = AT(I.z.zz, c0, k), z1 = AT(I.z.zz, c1, k);
  const float x0 = AT(I.b.s_exner, c0, k), x1 = AT(I.b.s_exner, c1, k);
  const float q0 = AT(I.b.rho_pp, c0, k), q1 = AT(I.b.rho_pp, c1, k);
  float to0 = 0.0f, to1 = 0.0f, st0 = 0.0f, st1 = 0.0f;
  if (DAMP) {
    if (!AVGRP) {  // after a stage's first substep (AVGRP: the second of two) rtheta_pp_old is zero
      to0 = AT(I.b.rtheta_pp_old, c0, k);
      to1 = AT(I.b.rtheta_pp_old, c1, k);
    }
    st0 = AT(I.b.s_theta, c0, k);
    st1 = AT(I.b.s_theta, c1, k);
  }
  const float ra_old = AVGRP ? rp_raw : ra_in;
  // ru_p + the divergence-damping increment (damped_ru_p's arithmetic)
  const float rp_in = DAMP ? rp_raw + ((damp_coef * ((tp0 - to0) - (tp1 - to1))) * (1.0f - 0.0f)) / (st0 + st1)
                           : rp_raw;
  float pg = ((tp1 - tp0) * idc) / (0.5f * (z1 + z0));
  pg = (((cqu * 0.5f) * I.k.c2) * (x0 + x1)) * pg;
  pg = pg + ((0.5f * zxu) * I.k.gravity) * (q0 + q1);
  const float p = rp_in + dts * (tr - pg);
  AT(I.b.ru_p, e, k) = p;
  AT(I.b.ru_avg, e, k) = ra_old + p;
}

// The acoustic column update (acoustic_v841.py:296-565) in three parts around
// the Thomas sweeps: the right-hand side, the Rayleigh damping and new
// perturbations, and (LAST) the recovery of the column.
// Level rows of a column block in LDS, in this order.
enum { LV_RDZW, LV_EWM, LV_EWP, LV_ETP, LV_ETM, LV_FZM, LV_FZP, LV_RDZU, LV_N };
// each wavefront of the block stages LV_PER of them
constexpr int LV_PER = LV_N / COLW_AC;
static_assert(LV_N % COLW_AC == 0, "level rows per wavefront");
__device__ __forceinline__ void level_rows(const Instance &I, int w, int k, float (&lv)[LV_PER]) {
  const float *const lev[LV_N] = {I.z.rdzw, I.z.ewm, I.z.ewp, I.z.etp, I.z.etm, I.z.fzm, I.z.fzp, I.z.rdzu};
#pragma unroll
  for (int j = 0; j < LV_PER; ++j) lv[j] = lev[w * LV_PER + j][k];
}
__device__ __forceinline__ void stage_level_rows(float *s_lev, int w, int k, const float (&lv)[LV_PER]) {
#pragma unroll
  for (int j = 0; j < LV_PER; ++j) s_lev[(w * LV_PER + j) * 64 + k] = lv[j];
}
template <int NE>
struct AcIn {
  float rpp, rtpp, rwp, wwa;            // zero at a stage's first substep
  float coftz, cofwt, cofwz, trho, trt, trw, zk, al, ga, srw, crw, damp, crho, wk, sthc;
  float rup[NE], sto[NE];               // ru_p of the cell's edges; start theta of the cells across them
};
struct AcMid {  // what the second part needs beside the column itself
  float rs, ts, wwa;
};
// returns the right-hand side and the sub-diagonal (times dts^2) of the column
template <int NE, bool FIRST>
__device__ __forceinline__ AcMid ac_rhs(const Instance &I, const AcIn<NE> &q, const float (&sg)[NE],
                                        const float (&sd)[NE], float ia, int n, int k, float dts, const float *lev,
                                        float &col, float &ad) {
  const int L = I.n.L;
  const float rdzw = lev[LV_RDZW * 64 + k], ewm = lev[LV_EWM * 64 + k], ewp = lev[LV_EWP * 64 + k];
  const float etp = lev[LV_ETP * 64 + k], etm = lev[LV_ETM * 64 + k], fzm = lev[LV_FZM * 64 + k];
  const float fzp = lev[LV_FZP * 64 + k];
  float r = 0.0f, t = 0.0f;
#pragma unroll
  for (int s = 0; s < NE; ++s)
    if (s < n) {
      // the first substep's ru_p is dts * tend_ru (the momentum pass's product)
      const float rp = FIRST ? dts * q.rup[s] : q.rup[s];
      const float flux = ((dts * sd[s]) * rp) * ia;  // (csign*dts)*dv, csign = +-1
      // theta at the edge: (theta[cell1] + theta[cell0]) in that order
      const bool first_cell = sg[s] > 0.0f;
      const float th0 = first_cell ? q.sthc : q.sto[s];
      const float th1 = first_cell ? q.sto[s] : q.sthc;
      r = r - flux;
      t = t - (flux * 0.5f) * (th1 + th0);
    }
  const float coftz_p = dn1(q.coftz);
  const float ewm_p = dn1(ewm);
  const float rwp_p = dn1(q.rwp);
  AcMid m;
  m.rs = ((q.rpp + dts * q.trho) + r) - (dts * rdzw) * (ewm_p * rwp_p - ewm * q.rwp);
  m.ts = ((q.rtpp + dts * q.trt) + t) - (dts * rdzw) * ((ewm_p * coftz_p) * rwp_p - (ewm * q.coftz) * q.rwp);
  m.wwa = q.wwa;
  if (k >= 1 && k < L) m.wwa = m.wwa + ewm * q.rwp;
  const float ts_m = up1(m.ts), rs_m = up1(m.rs), rtpp_m = up1(q.rtpp), rpp_m = up1(q.rpp), zk_m = up1(q.zk);
  const float cofwt_m = up1(q.cofwt);
  const float etp_m = up1(etp), etm_m = up1(etm);
  // cofwr and the sub-diagonal a of the implicit w system at levels 1..L-1,
  // formed from zz, the level rows and the coefficients of levels k and k-1
  // by the same operations as in coef_system
  const float rdzw_m = up1(rdzw), ewp_m = up1(ewp), coftz_m = up1(q.coftz);
  float cofwr = 0.0f, a = 0.0f;
  if (k >= 1 && k < L) {
    cofwr = (0.5f * I.k.gravity) * (fzm * q.zk + fzp * zk_m);
    a = (((-q.cofwz) * coftz_m) * rdzw_m) * zk_m + cofwr * rdzw_m - (cofwt_m * coftz_m) * rdzw_m;
    a = (a * etp_m) * ewp_m;
  }
  col = q.rwp;
  if (k >= 1 && k < L) {
    float x = q.trw -
              q.cofwz * (((etp * q.zk) * m.ts - (etp_m * zk_m) * ts_m) + ((etm * q.zk) * q.rtpp - (etm_m * zk_m) * rtpp_m));
    x = x - cofwr * ((etp * m.rs + etp_m * rs_m) + (etm * q.rpp + etm_m * rpp_m));
    x = x + q.cofwt * (etp * m.ts + etm * q.rtpp);
    x = x + cofwt_m * (etp_m * ts_m + etm_m * rtpp_m);
    col = col + dts * x;
  }
  const float dts2 = dts * dts;
  ad = dts2 * a;
  return m;
}
struct AcOut {
  float rwp, wwa, rpp, rtpp;
};
// the solved column: Rayleigh damping of w, then the new perturbations
__device__ __forceinline__ AcOut ac_update(const Instance &I, const AcMid &m, float col, float srw, float crw, float damp,
                                           float crho, float wk, float zk, float coftz, int k, float dts,
                                           const float *lev) {
  const int L = I.n.L;
  const float rdzw = lev[LV_RDZW * 64 + k], ewp = lev[LV_EWP * 64 + k];
  const float fzm = lev[LV_FZM * 64 + k], fzp = lev[LV_FZP * 64 + k];
  const float zk_m = up1(zk), crho_m = up1(crho), coftz_p = dn1(coftz), ewp_p = dn1(ewp);
  if (k >= 1 && k < L) {
    const float delta = srw - crw;
    const float zi = fzm * zk + fzp * zk_m;
    const float ri = fzm * crho + fzp * crho_m;
    col = (col + delta - (((dts * damp) * zi) * ri) * wk) / (1.0f + dts * damp) - delta;
  }
  AcOut o;
  o.wwa = m.wwa;
  if (k >= 1 && k < L) o.wwa = o.wwa + ewp * col;
  const float col_p = dn1(col);
  o.rwp = col;
  o.rpp = m.rs - (dts * rdzw) * (ewp_p * col_p - ewp * col);
  o.rtpp = m.ts - (dts * rdzw) * ((ewp_p * coftz_p) * col_p - (ewp * coftz) * col);
  return o;
}

// Recovery of a column after a stage's last substep (driver.py:3176-3290):
// rho, theta_m, rho*theta, the perturbations and rw; at stage 3 (S3) exner, p'
// and the split-transport sum of the vertical flux.  The column update holds
// the perturbations and rw, so recovering here saves storing them for the
// recovery pass and reading them back there and in the edge recovery (which
// reads the recovered rho instead of three rows per cell).
struct RecIn {
  float srp, rb, srtp, rtb, exb, spw;
};
template <bool S3>
__device__ __forceinline__ RecIn rec_rows(const Instance &I, int c, int k) {
  return {AT(I.b.s_rho_p, c, k),    AT(I.z.rb, c, k),
          AT(I.b.s_rtheta_p, c, k), AT(I.z.rtb, c, k),
          S3 ? AT(I.z.exb, c, k) : 0.0f, S3 ? AT(I.b.split_w, c, k) : 0.0f};
}
template <bool S3>
__device__ __forceinline__ void rec_column(const Instance &I, const RecIn &r, const AcOut &o, float srw, float zk, int c,
                                           int k, int sub, float inv_steps, int store_rtp) {
  const int L = I.n.L;
  const bool lay = k < L, inner = k >= 1 && k < L;
  const float dp = lay ? r.srp + o.rpp : 0.0f;
  const float rp = lay ? r.srtp + o.rtpp : 0.0f;
  const float rho = lay ? dp + r.rb : 1.0f;
  const float rtv = lay ? rp + r.rtb : 1.0f;
  int bad = (lay && (!(rho > 0.0f) || !(rtv > 0.0f))) ? 1 : 0;
  const float th = rtv / rho;
  float ex = 0.0f, ppv = 0.0f;
  if (S3 && lay) {
    const float arg = (zk * I.k.cfac) * rtv;
    if (!(arg > 0.0f)) bad = 1;
    ex = exner_pow(I, arg);
    ppv = (zk * I.k.rgas) * (ex * rp + r.rtb * (ex - r.exb));
  }
  if (lay) {
    AT(I.b.r_rho, c, k) = rho;
    AT(I.b.r_theta, c, k) = th;
    if (store_rtp) AT(I.b.r_rtheta_p, c, k) = rp;
    if (S3) {
      AT(I.b.r_rho_p, c, k) = dp;
      if (sub == I.k.splits) AT(I.b.r_rt, c, k) = rtv;  // read where the step publishes it only
      AT(I.b.r_exner, c, k) = ex;
      AT(I.b.r_pp, c, k) = ppv;
    }
  }
  if (k <= L) {
    AT(I.b.r_rw, c, k) = inner ? srw + o.rwp : 0.0f;
    if (S3) {
      const float fw = srw + o.wwa * inv_steps;
      const float acc = sub == 1 ? fw : fw + r.spw;
      AT(I.b.split_w, c, k) = sub == I.k.splits ? acc * I.k.split_inv : acc;
    }
  }
  if (bad) set_flag(I.b.flag);
}

// Scalars of a column pass that recovers its column.
struct RecArgs {
  int sub;          // dynamics subcycle
  float inv_steps;  // 1 / substeps of the stage
  int store_rtp;    // rtheta_p has a later reader
  int store_work;   // keep the working perturbations current (the step's last stage)
};

// FIRST: the first substep of a stage (the perturbation fields start at
// zero).  LAST: the stage's last substep on the whole-step path, which also
// recovers the column.  Every global load is issued before the column sweep.
template <int NE, bool FIRST, bool LAST, bool S3>
KBCOL(COLW_AC) k_ac_cell(const Instance I, float dts, int store_old, const RecArgs ra) {
  constexpr int COLW = COLW_AC;
  __shared__ float s_lev[LV_N * 64];
  const int w = (int)(threadIdx.x >> 6);
  const int c0 = wave_entity<COLW>();
  const bool live = c0 < I.n.C;
  const int c = live ? c0 : 0;  // every wave reaches the barriers
  const int k = lane();
  const int L = I.n.L;
  const int n = I.m.neoc[c];
  int e[NE], o[NE];
#pragma unroll
  for (int s = 0; s < NE; ++s) {
    e[s] = I.m.eoc[c * NE + s];
    o[s] = I.m.ocell[c * NE + s];  // the other cell of edge s
  }
  SlotRow<NE> sgr = slot_row<NE>(I.m.csign + c * NE), sdr = slot_row<NE>(I.m.csdv + c * NE);
  const float ia = uni_load(I.m.invarea + c);
  float lv[LV_PER];
  level_rows(I, w, k, lv);
  AcIn<NE> q;
  q.sthc = AT(I.b.s_theta, c, k);
  q.rpp = q.rtpp = q.rwp = q.wwa = 0.0f;
  if (!FIRST) {
    q.rpp = AT(I.b.rho_pp, c, k);
    q.rtpp = AT(I.b.rtheta_pp, c, k);
    q.rwp = AT(I.b.rw_p, c, k);
    q.wwa = AT(I.b.ww_avg, c, k);
  }
  q.coftz = AT(I.b.coftz, c, k);
  q.cofwt = AT(I.b.cofwt, c, k);
  q.cofwz = AT(I.b.cofwz, c, k);
  q.trho = AT(I.b.tend_rho, c, k);
  q.trt = AT(I.b.tend_rt, c, k);
  q.trw = AT(I.b.tend_rw, c, k);
  q.zk = AT(I.z.zz, c, k);
  q.al = AT(I.b.alpha, c, k);
  q.ga = AT(I.b.gamma, c, k);
  q.srw = AT(I.b.s_rw, c, k);
  q.crw = AT(I.b.c_rw, c, k);
  q.damp = AT(I.z.dss, c, k);
  q.crho = AT(I.b.c_rho, c, k);
  q.wk = AT(I.b.w, c, k);
#pragma unroll
  for (int s = 0; s < NE; ++s) {
    fence(e[s]);
    fence(o[s]);
  }
#pragma unroll
  for (int s = 0; s < NE; ++s) {
    q.rup[s] = FIRST ? AT(I.b.tend_ru, e[s], k) : AT(I.b.ru_p, e[s], k);
    q.sto[s] = AT(I.b.s_theta, o[s], k);
  }
  keep(q.rup, q.sto);
  stage_level_rows(s_lev, w, k, lv);
  settle(sgr, sdr);
  float sg[NE], sd[NE];
  slot_vals(sgr, sg);
  slot_vals(sdr, sd);
  __syncthreads();
  float col, ad;
  const AcMid m = ac_rhs<NE, FIRST>(I, q, sg, sd, ia, n, k, dts, s_lev, col, ad);
  RecIn r;
  if (LAST) r = rec_rows<S3>(I, c, k);  // in flight during the sweeps
  col = thomas_sweeps(col, ad, q.al, q.ga, k, L);
  const AcOut a =
      ac_update(I, m, col, q.srw, q.crw, q.damp, q.crho, q.wk, q.zk, q.coftz, k, dts, s_lev);
  if (!live) return;
  if (!LAST || ra.store_work) {
    if (k <= L) {
      AT(I.b.rw_p, c, k) = a.rwp;
      AT(I.b.ww_avg, c, k) = a.wwa;
    }
    if (k < L) AT(I.b.rho_pp, c, k) = a.rpp;
  }
  if (k < L) {
    AT(I.b.rtheta_pp, c, k) = a.rtpp;  // read by the damping that follows
    if (store_old) AT(I.b.rtheta_pp_old, c, k) = q.rtpp;
  }
  if (LAST) rec_column<S3>(I, r, a, q.srw, q.zk, c, k, ra.sub, ra.inv_steps, ra.store_rtp);
}

// A stage's column work in one pass on the whole-step path: (VC) the implicit
// coefficients, the theta and w tendencies, the first acoustic column update
// and (LAST, a stage of one substep) the recovery.  As passes of their own
// each of these reads the column's rows again (theta, zz, rw, w, tend_ru of
// the cell's edges) and hands its result over through memory (five
// coefficient rows, two tendencies, the perturbations).  x1.40962 moist, the
// stages of a subcycle with their recovery: 95 + 112 + 93 us against 168 + 182
// + 115 us in passes of their own (HBM-bound, 4.3-4.8 TB/s); x1.162, where
// each launch costs about 5 us: a whole step 662 -> 432 us with the side
// stream of the coefficients gone.
// The coefficients wait in LDS until the acoustic part, and its rows are loaded
// when the theta part has freed its registers.  Wavefronts per SIMD: as many as
// hold the pass without a vector register in memory, seven (six with coefficients
// and correction flux, or seven-edge cells; up to 34 scalar registers wait in lanes
// of vector registers); a CU then holds seven or six blocks of four columns, and
// the chains of some run under the loads of the others.  At eight wavefronts 3-11
// vector registers spill, and their traffic costs more than the occupancy gives: 119 + 166 + 112 us a subcycle's three stages at x1.40962
// against 95 + 116 + 93, both with the columns swept out of LDS (blocks of eight
// columns at six: 103 + 120 + 93).
template <int NE, bool VC, bool CORR, bool MIX, bool LAST, bool S3>
__global__ void __launch_bounds__(64 * COLW_AC)
    __attribute__((amdgpu_waves_per_eu(NE == 6 && !(VC && CORR) ? 7 : 6, NE == 6 && !(VC && CORR) ? 7 : 6)))
    k_col(const Instance I, float dts, const float *__restrict__ rtp, int store_old, int store_cof, int store_t,
      const RecArgs ra) {
  constexpr int COLW = COLW_AC;
  __shared__ float s_x[VC ? COLW * 64 : 1], s_l[COLW * 64], s_g[COLW * 64];
  __shared__ float s_cof[VC ? 3 * COLW * 64 : 1];  // coftz, cofwt, cofwz
  __shared__ float s_lev[LV_N * 64];
  const int w = (int)(threadIdx.x >> 6);
  const int c0 = wave_entity<COLW>();
  const bool live = c0 < I.n.C;
  const int c = live ? c0 : 0;  // every wave reaches the barriers
  const int k = lane();
  const int L = I.n.L;
  const int n = I.m.neoc[c];
  int e[NE], o[NE];
#pragma unroll
  for (int s = 0; s < NE; ++s) {
    e[s] = I.m.eoc[c * NE + s];
    o[s] = I.m.ocell[c * NE + s];  // the other cell of edge s
  }
  SlotRow<NE> sgr = slot_row<NE>(I.m.csign + c * NE), sdr = slot_row<NE>(I.m.csdv + c * NE);
  const float ia = uni_load(I.m.invarea + c);
  float lv[LV_PER];
  level_rows(I, w, k, lv);
  if (VC) {
    const CoefIn r = coef_rows(I, I.b.s_exner, I.b.theta, rtp, c, k);
    stage_level_rows(s_lev, w, k, lv);
    __syncthreads();
    const CoefOut cf = coef_system(I, r, k, s_lev[LV_FZM * 64 + k], s_lev[LV_FZP * 64 + k], s_lev[LV_RDZU * 64 + k],
                                   s_lev[LV_RDZW * 64 + k], s_lev[LV_ETP * 64 + k], s_lev[LV_EWP * 64 + k]);
    s_l[w * 64 + k] = cf.a;
    s_g[w * 64 + k] = cf.b;
    s_x[w * 64 + k] = cf.cc;
    s_cof[(0 * COLW + w) * 64 + k] = cf.coftz;
    s_cof[(1 * COLW + w) * 64 + k] = cf.cofwt;
    s_cof[(2 * COLW + w) * 64 + k] = cf.cofwz;
    hold_loads();
  } else {
    stage_level_rows(s_lev, w, k, lv);
  }
#pragma unroll
  for (int s = 0; s < NE; ++s) {
    fence(e[s]);
    fence(o[s]);
  }
  ThetaIn<NE> t;
  WIn<NE> v;
  AcIn<NE> q;
  theta_rows<NE, CORR, MIX>(I, e, c, k, t);
  if (!VC) w_rows<NE>(I, e, c, k, v);
  if (!VC) {
    __syncthreads();
  } else {
    float ca = s_l[w * 64 + k], cb = s_g[w * 64 + k];
    if (coef_sweep(ca, cb, s_x[w * 64 + k], k, L, dts * dts) && live) set_flag(I.b.flag);
    s_l[w * 64 + k] = ca;
    s_g[w * 64 + k] = cb;
    w_rows<NE>(I, e, c, k, v);
    if (live && store_cof)
      store_coefs(I, c, k, s_cof[(0 * COLW + w) * 64 + k], s_cof[(1 * COLW + w) * 64 + k],
                  s_cof[(2 * COLW + w) * 64 + k], 0.0f, ca, cb);
  }
  keep(t.fth);
  if (CORR) keep(t.fco);
  settle(sgr, sdr);
  float sg[NE], sd[NE];
  slot_vals(sgr, sg);
  slot_vals(sdr, sd);
  q.trt = theta_tendency<NE, CORR, MIX>(I, t, sg, ia, n, k, s_lev[LV_FZM * 64 + k], s_lev[LV_FZP * 64 + k],
                                        s_lev[LV_RDZW * 64 + k]);
  keep(q.trt);
  hold_loads();
  q.trho = AT(I.b.tend_rho, c, k);
  q.damp = AT(I.z.dss, c, k);
  q.crho = AT(I.b.c_rho, c, k);
#pragma unroll
  for (int s = 0; s < NE; ++s) q.sto[s] = AT(I.b.s_theta, o[s], k);
  keep(v.fwv, v.tru, v.zb, v.zb3);
  q.trw = w_tendency<NE>(I, v, t.rwc, sg, ia, n, k, s_lev[LV_FZM * 64 + k], s_lev[LV_FZP * 64 + k],
                         s_lev[LV_RDZU * 64 + k]);
  keep(q.trw);
  hold_loads();
  if (VC) {
    q.coftz = s_cof[(0 * COLW + w) * 64 + k];
    q.cofwt = s_cof[(1 * COLW + w) * 64 + k];
    q.cofwz = s_cof[(2 * COLW + w) * 64 + k];
  } else {
    q.coftz = AT(I.b.coftz, c, k);
    q.cofwt = AT(I.b.cofwt, c, k);
    q.cofwz = AT(I.b.cofwz, c, k);
    s_l[w * 64 + k] = AT(I.b.alpha, c, k);
    s_g[w * 64 + k] = AT(I.b.gamma, c, k);
  }
  if (live && store_t) store_tend(I, c, k, q.trt, q.trw);
  q.sthc = t.ths;
  q.rpp = q.rtpp = q.rwp = q.wwa = 0.0f;
  if (k >= L) q.trt = 0.0f;  // levels past the top read zero, as the stored rows hold
  q.zk = v.zz;
  q.srw = t.rws;
  q.crw = t.rwc;
  q.wk = v.ww;
#pragma unroll
  for (int s = 0; s < NE; ++s) q.rup[s] = v.tru[s];
  keep(q.sto);
  float col, ad;
  const AcMid m = ac_rhs<NE, true>(I, q, sg, sd, ia, n, k, dts, s_lev, col, ad);
  hold_loads();
  RecIn r;
  if (LAST) r = rec_rows<S3>(I, c, k);  // in flight during the sweeps
  col = thomas_sweeps(col, ad, s_l[w * 64 + k], s_g[w * 64 + k], k, L);
  const AcOut a =
      ac_update(I, m, col, q.srw, q.crw, q.damp, q.crho, q.wk, q.zk, q.coftz, k, dts, s_lev);
  if (!live) return;
  if (!LAST || ra.store_work) {
    if (k <= L) {
      AT(I.b.rw_p, c, k) = a.rwp;
      AT(I.b.ww_avg, c, k) = a.wwa;
    }
    if (k < L) AT(I.b.rho_pp, c, k) = a.rpp;
  }
  if (k < L) {
    AT(I.b.rtheta_pp, c, k) = a.rtpp;
    if (store_old) AT(I.b.rtheta_pp_old, c, k) = 0.0f;
  }
  if (LAST) rec_column<S3>(I, r, a, q.srw, q.zk, c, k, ra.sub, ra.inv_steps, ra.store_rtp);
}

KB k_divdamp(const Instance I, float coefficient) {
  const int e = wave_entity(I);
  if (e >= I.n.E) return;
  const int k = lane();
  if (k >= I.n.L) return;
  AT(I.b.ru_p, e, k) = damped_ru_p(I, e, k, AT(I.b.ru_p, e, k), coefficient);
}

// --------------------------------------------------------------------- recovery
// w from rw and the terrain-following horizontal flux (terrain.py:491-571) of
// the edge momentum ru, and (hdiv_out) its mass-flux divergence.
template <int NE>
struct RecWIn {
  float ru[NE], zb[NE], zb3[NE];
  SlotRow<NE> sg, sd;
  float ia, zk, fzm, fzp;
  int n, e[NE];
};
template <int NE>
__device__ __forceinline__ void rec_w_index(const Instance &I, int c, int k, RecWIn<NE> &a) {
  a.n = I.m.neoc[c];
#pragma unroll
  for (int s = 0; s < NE; ++s) a.e[s] = I.m.eoc[c * NE + s];
  a.sg = slot_row<NE>(I.m.csign + c * NE);
  a.sd = slot_row<NE>(I.m.csdv + c * NE);
  a.ia = uni_load(I.m.invarea + c);
  a.zk = AT(I.z.zz, c, k);
  a.fzm = AT(I.z.fzm, 0, k);
  a.fzp = AT(I.z.fzp, 0, k);
#pragma unroll
  for (int s = 0; s < NE; ++s) {
    a.zb[s] = AT(I.z.zb, c * NE + s, k);
    a.zb3[s] = AT(I.z.zb3, c * NE + s, k);
  }
}
template <int NE>
__device__ __forceinline__ void rec_w_fence(const RecWIn<NE> &a) {
#pragma unroll
  for (int s = 0; s < NE; ++s) fence(a.e[s]);
}
template <int NE>
__device__ __forceinline__ void rec_w_rows(const Instance &I, const float *ru, int k, RecWIn<NE> &a) {
#pragma unroll
  for (int s = 0; s < NE; ++s) a.ru[s] = AT(ru, a.e[s], k);
}
template <int NE, bool HDIV>
__device__ __forceinline__ float rec_w_compute(const Instance &I, int k, const RecWIn<NE> &a, float rho_k, float rw_k,
                                               float &hdiv) {
  const int L = I.n.L, n = a.n;
  float sg[NE];
#pragma unroll
  for (int s = 0; s < NE; ++s) sg[s] = a.sg[s];
  const float zkm = up1(a.zk);
  if (HDIV) {
    // mass-flux divergence of the recovered ru (dynamics.py:86-121), next stage's hdiv
    float acc = 0.0f;
#pragma unroll
    for (int s = 0; s < NE; ++s)
      if (s < n) acc = acc + a.sd[s] * a.ru[s];
    hdiv = acc * a.ia;
  }
  float col = 0.0f;
  if (k >= 1 && k < L) col = rw_k / (a.fzm * a.zk + a.fzp * zkm);
  const float cf1 = I.z.cf1, cf2 = I.z.cf2, cf3 = I.z.cf3;
#pragma unroll
  for (int s = 0; s < NE; ++s) {
    const float ru_m = up1(a.ru[s]);
    const float ru0 = rdl(a.ru[s], 0), ru1 = rdl(a.ru[s], 1), ru2 = rdl(a.ru[s], 2);
    if (s < n) {
      if (k == 0) {
        const float flux = (cf1 * ru0 + cf2 * ru1) + cf3 * ru2;
        col = col + (sg[s] * (a.zb[s] + cs1(flux) * a.zb3[s])) * flux;
      } else if (k < L) {
        const float flux = a.fzm * a.ru[s] + a.fzp * ru_m;
        col = col + (sg[s] * (a.zb[s] + cs1(flux) * a.zb3[s])) * flux;
      }
    }
  }
  const float r0 = rdl(rho_k, 0), r1 = rdl(rho_k, 1), r2 = rdl(rho_k, 2);
  const float rho_m = up1(rho_k);
  if (k == 0) {
    const float bottom = (cf1 * r0 + cf2 * r1) + cf3 * r2;
    col = col / bottom;
  } else if (k < L) {
    col = col / (a.fzm * rho_k + a.fzp * rho_m);
  } else {
    col = 0.0f;
  }
  return col;
}
template <int NE, bool HDIV>
__device__ __forceinline__ float recover_w_column(const Instance &I, int c, int k, float rho_k, float rw_k,
                                                  const float *ru, float &hdiv) {
  RecWIn<NE> a;
  rec_w_index(I, c, k, a);
  rec_w_fence(a);
  rec_w_rows(I, ru, k, a);
  keep(a.ru, a.zb, a.zb3);
  settle(a.sg, a.sd);
  return rec_w_compute<NE, HDIV>(I, k, a, rho_k, rw_k, hdiv);
}

// The part of a recovery that reads the cell's recovered edges, after a column
// pass that recovered the column: terrain w and (HDIV) the next stage's
// mass-flux divergence.  After stage 3 the next subcycle's opening pass forms
// the divergence again.
// DIAG: also the cell and vertex diagnostics of the recovered u, which read
// the same edges: one batch of loads and one launch instead of two (55 us
// against 34 + 34 at x1.40962).
template <int NE, bool HDIV, bool DIAG>
__device__ __forceinline__ void rec_w_cell(const Instance &I, int c, int k, int store_mix) {
  const float rho = AT(I.b.c_rho, c, k), rwv = AT(I.b.c_rw, c, k);
  RecWIn<NE> a;
  CellVertIn<NE> d;
  rec_w_index(I, c, k, a);
  if (DIAG) cell_vert_index(I, c, d);
  rec_w_fence(a);
  if (DIAG) cell_vert_fence(d);
  rec_w_rows(I, I.b.c_ru, k, a);
  if (DIAG) cell_vert_rows(I, I.b.u, k, d);
  keep(a.ru, a.zb, a.zb3);
  settle(a.sg, a.sd);
  float hd = 0.0f;
  const float wv = rec_w_compute<NE, HDIV>(I, k, a, rho, rwv, hd);
  if (DIAG) {
    keep(d.uo, d.ux, d.ia);
    settle(d.sd, d.dd, d.kt, d.rec);
  }
  if (HDIV && k < I.n.L) AT(I.b.hdiv, c, k) = hd;
  if (k <= I.n.L) AT(I.b.w, c, k) = wv;
  if (DIAG) cell_vert_finish(I, c, k, d, store_mix);
}
template <int NE, bool HDIV, bool DIAG>
KB k_rec_w(const Instance I, int store_mix) {
  const int c = wave_entity(I);
  if (c < I.n.C) rec_w_cell<NE, HDIV, DIAG>(I, c, lane(), store_mix);
}

// The whole cell recovery as a pass of its own (the phase entry points).
// S3: the stage-3 recovery (exner, p' and the split-transport sums).  The
// loads and the terrain w recovery come first, branch-free, so every gather
// of the pass is in flight together; stores come last.
template <int NE, bool S3>
KB k_rec_cell(const Instance I, int sub, float inv_steps) {
  const int c = wave_entity(I);
  if (c >= I.n.C) return;
  const int k = lane();
  const int L = I.n.L;
  const bool lay = k < L, itf = k <= L, inner = k >= 1 && k < L;
  const float srp = AT(I.b.s_rho_p, c, k), rpp = AT(I.b.rho_pp, c, k);
  const float srtp = AT(I.b.s_rtheta_p, c, k), rtpp = AT(I.b.rtheta_pp, c, k);
  const float rb = AT(I.z.rb, c, k), rtb = AT(I.z.rtb, c, k);
  const float srw = AT(I.b.s_rw, c, k), rwp = AT(I.b.rw_p, c, k), wwa = AT(I.b.ww_avg, c, k);
  float zk = 0.0f, exb = 0.0f, spw = 0.0f;
  if (S3) {
    zk = AT(I.z.zz, c, k);
    exb = AT(I.z.exb, c, k);
    spw = AT(I.b.split_w, c, k);
  }
  const float dp = lay ? srp + rpp : 0.0f;
  const float rp = lay ? srtp + rtpp : 0.0f;
  const float rho = lay ? dp + rb : 1.0f;
  const float rtv = lay ? rp + rtb : 1.0f;
  const float rwv = inner ? srw + rwp : 0.0f;
  float hd = 0.0f;
  // hdiv feeds the next stage's momentum tendency; after stage 3 the next
  // subcycle's opening pass forms it again
  const float wv = recover_w_column<NE, !S3>(I, c, k, rho, rwv, I.b.c_ru, hd);
  int bad = (lay && (!(rho > 0.0f) || !(rtv > 0.0f))) ? 1 : 0;
  const float th = rtv / rho;
  float ex = 0.0f, ppv = 0.0f;
  if (S3 && lay) {
    const float arg = (zk * I.k.cfac) * rtv;
    if (!(arg > 0.0f)) bad = 1;
    ex = exner_pow(I, arg);
    ppv = (zk * I.k.rgas) * (ex * rp + rtb * (ex - exb));
  }
  const float fw = srw + wwa * inv_steps;
  float split = 0.0f;
  if (S3) {
    // split-transport sums: copy, then accumulate; the last subcycle also
    // applies the 1/splits average (integration.py:27-82)
    const float acc = sub == 1 ? fw : fw + spw;
    split = sub == I.k.splits ? acc * I.k.split_inv : acc;
  }
  if (lay) {
    AT(I.b.rho_p, c, k) = dp;
    AT(I.b.c_rt, c, k) = rtv;
    AT(I.b.rtheta_p, c, k) = rp;
    AT(I.b.c_rho, c, k) = rho;
    AT(I.b.theta, c, k) = th;
    if (S3) {
      AT(I.b.exner, c, k) = ex;
      AT(I.b.pp, c, k) = ppv;
    }
    if (!S3) AT(I.b.hdiv, c, k) = hd;
  }
  if (itf) {
    AT(I.b.c_rw, c, k) = rwv;
    AT(I.b.flux_w, c, k) = fw;
    if (S3) AT(I.b.split_w, c, k) = split;
    AT(I.b.w, c, k) = wv;
  }
  if (bad) set_flag(I.b.flag);
}

// DAMP: apply the last substep's divergence damping to ru_p first.
// AVGRP: one substep and ru_avg not stored, so the average is the undamped
// ru_p of that substep.  S3: accumulate the split-transport sums.  RHO: the
// column pass has recovered rho.  Loads first, stores last.
template <bool S3, bool DAMP, bool AVGRP, bool RHO>
KB k_rec_edge(const Instance I, int sub, float inv_steps, float damp_coef, float dts) {
  const int e = wave_entity(I);
  if (e >= I.n.E) return;
  const int k = lane();
  if (k >= I.n.L) return;
  const int c0 = I.m.coe[2 * e], c1 = I.m.coe[2 * e + 1];
  const float sru = AT(I.b.s_ru, e, k);
  // one substep: its ru_p is dts * tend_ru, formed here as the momentum pass formed it
  const float rp_ld = AVGRP ? AT(I.b.tend_ru, e, k) : AT(I.b.ru_p, e, k);
  const float avg_ld = AVGRP ? 0.0f : AT(I.b.ru_avg, e, k);
  const float spu = S3 ? AT(I.b.split_u, e, k) : 0.0f;
  const float r0 = RHO ? AT(I.b.c_rho, c0, k) : (AT(I.b.s_rho_p, c0, k) + AT(I.b.rho_pp, c0, k)) + AT(I.z.rb, c0, k);
  const float r1 = RHO ? AT(I.b.c_rho, c1, k) : (AT(I.b.s_rho_p, c1, k) + AT(I.b.rho_pp, c1, k)) + AT(I.z.rb, c1, k);
  const float rp_raw = AVGRP ? dts * rp_ld : rp_ld;
  const float avg = AVGRP ? rp_raw : avg_ld;
  const float rp = DAMP ? damped_ru_p<AVGRP>(I, e, k, rp_raw, damp_coef) : rp_raw;
  const float ru = sru + rp;
  const float fu = sru + avg * inv_steps;
  float split = 0.0f;
  if (S3) {
    const float acc = sub == 1 ? fu : fu + spu;
    split = sub == I.k.splits ? acc * I.k.split_inv : acc;
  }
  const float uu = (2.0f * ru) / (r0 + r1);
  // the damped ru_p is read again only as the step's output (stage 3) or by
  // an export between phases; the next stage forms its own
  if (DAMP && (S3 || I.k.store_flux)) AT(I.b.ru_p, e, k) = rp;
  AT(I.b.c_ru, e, k) = ru;
  if (I.k.store_flux) AT(I.b.flux_u, e, k) = fu;
  if (S3) AT(I.b.split_u, e, k) = split;
  AT(I.b.u, e, k) = uu;
}

// rebuild of the saved diagnostics from a prognostic state (driver.py:2655-2700)
template <int NE>
KB k_rebuild_cell(const Instance I) {
  const int c = wave_entity(I);
  if (c >= I.n.C) return;
  const int k = lane();
  const int L = I.n.L;
  // every load before any store (the terrain w recovery gathers among them)
  const float rho_k = AT(I.b.rho, c, k), rt = AT(I.b.rt, c, k), zk = AT(I.z.zz, c, k);
  const float rtb = AT(I.z.rtb, c, k), rb = AT(I.z.rb, c, k), exb = AT(I.z.exb, c, k);
  const float rwk = AT(I.b.rw, c, k);
  const float rho = k < L ? rho_k : 1.0f;
  float hd;
  const float wv = recover_w_column<NE, false>(I, c, k, rho, rwk, I.b.ru, hd);
  if (k < L) {
    const float ex = exner_pow(I, (zk * I.k.cfac) * rt);
    const float rtp = rt - rtb;
    AT(I.b.theta, c, k) = rt / rho;
    AT(I.b.exner, c, k) = ex;
    AT(I.b.rho_p, c, k) = rho - rb;
    AT(I.b.rtheta_p, c, k) = rtp;
    AT(I.b.pp, c, k) = (zk * I.k.rgas) * (ex * rtp + rtb * (ex - exb));
  }
  if (k <= L) AT(I.b.w, c, k) = wv;
}

KB k_rebuild_edge(const Instance I) {
  const int e = wave_entity(I);
  if (e >= I.n.E) return;
  const int k = lane();
  if (k >= I.n.L) return;
  const int c0 = I.m.coe[2 * e], c1 = I.m.coe[2 * e + 1];
  AT(I.b.u, e, k) = (2.0f * AT(I.b.ru, e, k)) / (AT(I.b.rho, c0, k) + AT(I.b.rho, c1, k));
}

// ------------------------------------------------------------ scalar transport
// q0..q3: the column's values at levels k-2, k-1, k, k+1
__device__ __forceinline__ float vflux(float q0, float q1, float q2, float q3, float wk, int k, int L, float fzm,
                                       float fzp, float coef) {
  if (k == 1 || k == L - 1) return wk * (fzm * q2 + fzp * q1);
  const float base = div12(wk * (7.0f * (q2 + q1) - (q3 + q0)));
  const float corr = div12((coef * fabsf(wk)) * ((q3 - q0) - 3.0f * (q2 - q1)));
  return base + corr;
}

// Scalar kernels run one wavefront per entity over all species: the
// connectivity, stencil weights and the species-independent rows are read
// once, and the species are taken in batches of G whose rows are all
// requested before any of them is combined (each batch is one memory round
// trip; a batch's stores come after its loads, and the next batch's loads
// after those stores, since the kernels' input and output arrays may alias).
// G trades round trips against registers per wavefront.
#ifndef HEXDYN_G_SC_EDGE
#define HEXDYN_G_SC_EDGE 3
#endif
#ifndef HEXDYN_G_SC_CELL
#define HEXDYN_G_SC_CELL 3
#endif
#ifndef HEXDYN_G_FCT_EDGE1
#define HEXDYN_G_FCT_EDGE1 6  // every species in one batch: 152 us against 158 us in batches of 3 (x1.40962)
#endif
#ifndef HEXDYN_G_FCT_CELL1
#define HEXDYN_G_FCT_CELL1 2
#endif
#ifndef HEXDYN_G_FCT_CELL2
#define HEXDYN_G_FCT_CELL2 2
#endif
__device__ __forceinline__ int clamp_sp(int sp, int nt) { return sp < nt ? sp : nt - 1; }

template <int NE>
__device__ __forceinline__ void sc_edge(const Instance &I, int e, int k, const float *__restrict__ qs,
                                        float *__restrict__ ev) {
  constexpr int NX = 2 * NE - 2, G = HEXDYN_G_SC_EDGE;
  const int NT = I.n.NT;
  int ac[NX];
#pragma unroll
  for (int s = 0; s < NX; ++s) ac[s] = I.m.advc[e * NX + s];
  const int na = I.m.nadv[e];
  SlotRow<NX> av = slot_row<NX>(I.m.adv + e * NX), a3v = slot_row<NX>(I.m.adv3 + e * NX);
  const float uu = AT(I.b.split_u, e, k);
#pragma unroll
  for (int s = 0; s < NX; ++s) fence(ac[s]);
  const float coef = I.k.coef3;
  for (int sp0 = (int)blockIdx.y * G; sp0 < NT; sp0 += (int)gridDim.y * G) {
    float v[G][NX];
#pragma unroll
    for (int g = 0; g < G; ++g) {
      const int r0 = clamp_sp(sp0 + g, NT) * I.n.C;  // species rows start at s * C
#pragma unroll
      for (int s = 0; s < NX; ++s) v[g][s] = AT(qs, r0 + ac[s], k);
    }
    // the weights are formed after the batch's loads are issued
    float uk = uu;
    keep(uk);
    keep(v);
    SlotRow<NX> avs = av, a3s = a3v;
    settle(avs, a3s);
    const float sv = cs1(uk);
    float wt[NX];
#pragma unroll
    for (int s = 0; s < NX; ++s) wt[s] = avs[s] + (coef * sv) * a3s[s];
#pragma unroll
    for (int g = 0; g < G; ++g) {
      if (sp0 + g >= NT) break;
      float r = 0.0f;
#pragma unroll
      for (int s = 0; s < NX; ++s)
        if (s < na) r = r + wt[s] * v[g][s];
      if (k < I.n.L) AT(ev, (sp0 + g) * I.n.E + e, k) = r;
    }
  }
}

template <int NE>
KB k_sc_edge(const Instance I, const float *__restrict__ qs, float *__restrict__ ev) {
  const int e = wave_entity(I);
  if (e < I.n.E) sc_edge<NE>(I, e, lane(), qs, ev);
}
// The transport's first edge pass and the recovery of w that ends the dynamics,
// neither of which reads what the other writes, in one launch where both
// together are small (HX_SMALL: meshes of 642 cells take it, 2562 do not): a
// x1.162 step 288 -> 281 us.  On large meshes the shared launch is slower than
// the two (174.5 us against 122.2 + 36.8 at x1.40962, 40.6 against 29.5 + 10.2 at
// x1.10242).
template <int NE>
KB k_sc_edge_w(const Instance I, int nb0, const float *__restrict__ qs, float *__restrict__ ev) {
  if ((int)blockIdx.x < nb0) {
    const int e = wave_entity_first(I, nb0);
    if (e < I.n.E) sc_edge<NE>(I, e, lane(), qs, ev);
  } else if (blockIdx.y == 0) {
    const int c = wave_entity_second(I, nb0);
    if (c < I.n.C) rec_w_cell<NE, false, false>(I, c, lane(), 0);
  }
}

template <int NE>
KB k_sc_cell(const Instance I, const float *__restrict__ qs, const float *__restrict__ ev, float *__restrict__ out,
             float dt, float wn, const float *__restrict__ src) {
  constexpr int G = HEXDYN_G_SC_CELL;
  const int c = wave_entity(I);
  if (c >= I.n.C) return;
  const int k = lane();
  const int L = I.n.L, NT = I.n.NT;
  const int n = I.m.neoc[c];
  int e[NE];
#pragma unroll
  for (int s = 0; s < NE; ++s) e[s] = I.m.eoc[c * NE + s];
  SlotRow<NE> sgr = slot_row<NE>(I.m.csign + c * NE);
  const float ia = uni_load(I.m.invarea + c);
  const float sw = AT(I.b.split_w, c, k);
  const float orho = AT(I.b.rho, c, k), crho = AT(I.b.c_rho, c, k);
  const float fzm = AT(I.z.fzm, 0, k), fzp = AT(I.z.fzp, 0, k), rdzw = AT(I.z.rdzw, 0, k);
#pragma unroll
  for (int s = 0; s < NE; ++s) fence(e[s]);
  float uh[NE];
#pragma unroll
  for (int s = 0; s < NE; ++s) uh[s] = AT(I.b.split_u, e[s], k);
  for (int sp0 = (int)blockIdx.y * G; sp0 < NT; sp0 += (int)gridDim.y * G) {
    float qk[G], qo[G], sr[G], evv[G][NE];
#pragma unroll
    for (int g = 0; g < G; ++g) {
      const int sq = clamp_sp(sp0 + g, NT);
      qk[g] = AT(qs, sq * I.n.C + c, k);
      qo[g] = AT(I.b.q, sq * I.n.C + c, k);
#pragma unroll
      for (int s = 0; s < NE; ++s) evv[g][s] = AT(ev, sq * I.n.E + e[s], k);
    }
    // held scalar tendency (transport.py:1800-1808)
#pragma unroll
    for (int g = 0; g < G; ++g) sr[g] = src ? AT(src, clamp_sp(sp0 + g, NT) * I.n.C + c, k) : 0.0f;
    keep(qk, qo, evv);
    keep(uh);
    SlotRow<NE> sgs = sgr;
    settle(sgs);
    float sg[NE];
    slot_vals(sgs, sg);
    const float target = (1.0f - wn) * orho + wn * crho;
#pragma unroll
    for (int g = 0; g < G; ++g) {
      if (sp0 + g >= NT) break;
      const float q_m2 = up1(up1(qk[g])), q_m1 = up1(qk[g]), q_p1 = dn1(qk[g]);
      float vf = 0.0f;
      if (k >= 1 && k < L) vf = vflux(q_m2, q_m1, qk[g], q_p1, sw, k, L, fzm, fzp, I.k.coef3);
      const float vf_p = dn1(vf);
      float tc = 0.0f;
#pragma unroll
      for (int s = 0; s < NE; ++s)
        if (s < n) tc = tc + ((-sg[s]) * uh[s]) * evv[g][s];
      tc = tc * ia + sr[g];
      if (k < L) {
        const float num = qo[g] * orho + dt * (tc - rdzw * (vf_p - vf));
        AT(out, (sp0 + g) * I.n.C + c, k) = num * (1.0f / target);
      }
    }
  }
}

// old mixing ratio with the held scalar tendency, old + dt*source/rho_old
// (transport.py:1906), every species of cell c
KB k_fct_source(const Instance I, float dt) {
  const int c = wave_entity(I);
  if (c >= I.n.C) return;
  const int k = lane();
  if (k >= I.n.L) return;
  const float rho = AT(I.b.rho, c, k);
  const int NT = I.n.NT;
  for (int s0 = 0; s0 < NT; s0 += HX_MOIST_G) {  // every row of a batch loaded before its stores
    float q[HX_MOIST_G], f[HX_MOIST_G];
#pragma unroll
    for (int g = 0; g < HX_MOIST_G; ++g) {
      const int r = (s0 + g < NT ? s0 + g : NT - 1) * I.n.C + c;
      q[g] = AT(I.b.q, r, k);
      f[g] = AT(I.b.phys_q, r, k);
    }
    keep(q, f);
#pragma unroll
    for (int g = 0; g < HX_MOIST_G; ++g)
      if (s0 + g < NT) AT(I.b.q_src, (s0 + g) * I.n.C + c, k) = q[g] + (dt * f[g]) / rho;
  }
}


template <int NE>
KB k_fct_edge1(const Instance I, const float *__restrict__ qs, float dt, const float *__restrict__ qold, float qadd) {
  constexpr int NX = 2 * NE - 2, G = HEXDYN_G_FCT_EDGE1;
  const int e = wave_entity(I);
  if (e >= I.n.E) return;
  const int k = lane();
  const int NT = I.n.NT;
  int ac[NX];
#pragma unroll
  for (int s = 0; s < NX; ++s) ac[s] = I.m.advc[e * NX + s];
  const int c1 = I.m.coe[2 * e], c2 = I.m.coe[2 * e + 1];
  const int na = I.m.nadv[e];
  SlotRow<NX> av = slot_row<NX>(I.m.adv + e * NX), a3v = slot_row<NX>(I.m.adv3 + e * NX);
  const float dve = uni_load(I.m.dv + e);
  const float uu = AT(I.b.split_u, e, k);
#pragma unroll
  for (int s = 0; s < NX; ++s) fence(ac[s]);
  fence(c1);
  fence(c2);
  const float coef = I.k.coef3;
  const float dvdt = dve * dt;
  for (int sp0 = (int)blockIdx.y * G; sp0 < NT; sp0 += (int)gridDim.y * G) {
    float v[G][NX], q1[G], q2[G];
#pragma unroll
    for (int g = 0; g < G; ++g) {
      const int p = clamp_sp(sp0 + g, NT) * I.n.C;
#pragma unroll
      for (int s = 0; s < NX; ++s) v[g][s] = AT(qs, p + ac[s], k);
      q1[g] = AT(qold, p + c1, k);
      q2[g] = AT(qold, p + c2, k);
    }
    float uk = uu;
    keep(uk);
    keep(v);
    SlotRow<NX> avs = av, a3s = a3v;
    settle(avs, a3s);
    const float sv = cs1(uk);
    float wt[NX];
#pragma unroll
    for (int s = 0; s < NX; ++s) wt[s] = avs[s] + (coef * sv) * a3s[s];
#pragma unroll
    for (int g = 0; g < G; ++g) {
      if (sp0 + g >= NT) break;
      const float qa1 = q1[g] + qadd, qa2 = q2[g] + qadd;
      float ra;
      if (na == 10) {
        // ten-cell stencils associate from the first product (transport.py n_adv == 10 branch)
        float xa = wt[0] * v[g][0];
#pragma unroll
        for (int s = 1; s < NX; ++s)
          if (s < 10) xa = xa + wt[s] * v[g][s];
        ra = uk * xa;
      } else {
        ra = 0.0f;
#pragma unroll
        for (int s = 0; s < NX; ++s)
          if (s < na) ra = ra + (uk * wt[s]) * v[g][s];
      }
      const float upa = dvdt * (max0(uk) * qa1 + min0(uk) * qa2);  // formed again by k_fct_cell1
      if (k < I.n.L) AT(I.b.fct_hres, (sp0 + g) * I.n.E + e, k) = dt * ra - upa;
    }
  }
}

// The upwind flux of each edge, dv*dt*(max(u,0)*q[cell0] + min(u,0)*q[cell1])
// (k_fct_edge1 forms the same value for the high-order residual), is formed
// here from the edge's split u and the old mixing ratios of its two cells,
// which the bounds read anyway: one u row per edge instead of one flux row
// per edge and species.  PAIR: cellsOnCell slot s is the other cell of
// edgesOnCell slot s in every cell (as in MPAS meshes); otherwise that cell's
// row is read separately.
template <int NE, bool PAIR>
KB k_fct_cell1(const Instance I, const float *__restrict__ qs, float dt, const float *__restrict__ qold, float qadd) {
  constexpr int G = HEXDYN_G_FCT_CELL1, NP = PAIR ? 1 : NE;
  const int c = wave_entity(I);
  if (c >= I.n.C) return;
  const int k = lane();
  const int L = I.n.L, NT = I.n.NT;
  const int n = I.m.neoc[c];
  int nb[NE], e[NE], oc[NP];
#pragma unroll
  for (int s = 0; s < NE; ++s) {
    nb[s] = I.m.coc[c * NE + s];
    e[s] = I.m.eoc[c * NE + s];
    if (!PAIR) oc[s < NP ? s : 0] = I.m.ocell[c * NE + s];
  }
  SlotRow<NE> sgr = slot_row<NE>(I.m.csign + c * NE), sdr = slot_row<NE>(I.m.csdv + c * NE);
  const float ia = uni_load(I.m.invarea + c);
  const float orho = AT(I.b.rho, c, k);
  const float wk = AT(I.b.split_w, c, k);
  const float rdzw = AT(I.z.rdzw, 0, k), fzm = AT(I.z.fzm, 0, k), fzp = AT(I.z.fzp, 0, k);
#pragma unroll
  for (int s = 0; s < NE; ++s) {
    fence(nb[s]);
    fence(e[s]);
  }
  if (!PAIR)
#pragma unroll
    for (int s = 0; s < NP; ++s) fence(oc[s]);
  float uh[NE];
#pragma unroll
  for (int s = 0; s < NE; ++s) uh[s] = AT(I.b.split_u, e[s], k);
  for (int sp0 = (int)blockIdx.y * G; sp0 < NT; sp0 += (int)gridDim.y * G) {
    float qsk[G], qol[G], qn[G][NE], qp[G][NP], hres[G][NE];
#pragma unroll
    for (int g = 0; g < G; ++g) {
      const int sq = clamp_sp(sp0 + g, NT);
      const int po = sq * I.n.C;
      qsk[g] = AT(qs, po + c, k);
#pragma unroll
      for (int s = 0; s < NE; ++s) {
        qn[g][s] = AT(qold, po + nb[s], k);
        hres[g][s] = AT(I.b.fct_hres, sq * I.n.E + e[s], k);
      }
      if (!PAIR)
#pragma unroll
        for (int s = 0; s < NP; ++s) qp[g][s] = AT(qold, po + oc[s], k);
      qol[g] = AT(qold, po + c, k);
    }
    keep(qsk, qol, qn, hres, uh);
    if (!PAIR) keep(qp);
    SlotRow<NE> sgs = sgr, sds = sdr;
    settle(sgs, sds);
    float sg[NE], sd[NE];
    slot_vals(sgs, sg);
    slot_vals(sds, sd);
    // the target density (transport.py:1964-1989): the old density plus dt
    // times the split mass-flux convergence, from rows this pass holds; the
    // first batch stores it for the second pass and checks it
    float hd = 0.0f;
#pragma unroll
    for (int s = 0; s < NE; ++s)
      if (s < n) hd = hd + (-(uh[s] * sd[s])) * ia;  // ((-csign)*uh)*dv, csign = +-1
    const float wk_p = dn1(wk);
    const float target = orho + dt * (hd - rdzw * (wk_p - wk));
    if (sp0 == 0 && k < L) {
      AT(I.b.target, c, k) = target;
      if (!(target > 0.0f)) set_flag(I.b.flag);
    }
#pragma unroll
    for (int g = 0; g < G; ++g) {
      if (sp0 + g >= NT) break;
      const int sp = sp0 + g;
      const float qs_k = qsk[g];
      const float qs_m2 = up1(up1(qs_k)), qs_m1 = up1(qs_k), qs_p1 = dn1(qs_k);
      const float qo = qol[g] + qadd;
      const float qo_m = up1(qo), qo_p = dn1(qo);
      float a, b;
      if (k == 0) {
        a = qo; b = qo;
        a = pmin(a, qo_p); b = pmax(b, qo_p);
      } else if (k == L - 1) {
        a = qo_m; b = qo_m;
        a = pmin(a, qo); b = pmax(b, qo);
      } else {
        a = qo_m; b = qo_m;
        a = pmin(a, qo); b = pmax(b, qo);
        a = pmin(a, qo_p); b = pmax(b, qo_p);
      }
#pragma unroll
      for (int s = 0; s < NE; ++s)
        if (s < n) {
          const float q = qn[g][s] + qadd;
          a = pmin(a, q);
          b = pmax(b, q);
        }
      float mass = qo * orho;
      float vres = 0.0f;
      float fcol = 0.0f;
      if (k >= 1 && k < L) {
        vres = dt * vflux(qs_m2, qs_m1, qs_k, qs_p1, wk, k, L, fzm, fzp, I.k.coef3);
        fcol = dt * (max0(wk) * qo_m + min0(wk) * qo);
      } else {
        vres = dt * 0.0f;
      }
      const float fcol_p = dn1(fcol);
      if (k <= L - 2) mass = mass - fcol_p * rdzw;
      if (k >= 1 && k < L) {
        mass = mass + fcol * rdzw;
        vres = vres - fcol;
      }
      const float vres_p = dn1(vres);
      float sin_ = (-rdzw) * (min0(vres_p) - max0(vres));
      float sout = (-rdzw) * (max0(vres_p) - min0(vres));
#pragma unroll
      for (int s = 0; s < NE; ++s)
        if (s < n) {
          const float so = -sg[s];
          // edge s's cells in edge order: this one first where csign = +1
          const float qx = (PAIR ? qn[g][s] : qp[g][s < NP ? s : 0]) + qadd;
          const bool first = sg[s] > 0.0f;
          const float qa1 = first ? qo : qx, qa2 = first ? qx : qo;
          const float dvdt = __builtin_fabsf(sd[s]) * dt;  // |csign * dv| = dv
          const float upa = dvdt * (max0(uh[s]) * qa1 + min0(uh[s]) * qa2);
          mass = mass + (so * upa) * ia;
          const float sr = (-so) * hres[g][s];
          sout = sout - max0(sr) * ia;
          sin_ = sin_ - min0(sr) * ia;
        }
      float f = (b * target - mass) / (sin_ + 1.0e-20f);
      sin_ = pmin(1.0f, max0(f));
      f = (a * target - mass) / (sout - 1.0e-20f);
      sout = pmin(1.0f, max0(f));
      if (k < L) {
        AT(I.b.fct_mass, sp * I.n.C + c, k) = mass;
        AT(I.b.fct_sin, sp * I.n.C + c, k) = sin_;
        AT(I.b.fct_sout, sp * I.n.C + c, k) = sout;
      }
      if (k <= L) AT(I.b.fct_vres, sp * I.n.C + c, k) = vres;
    }
  }
}

// The limited update of a cell.  Each edge's limited flux
// max(f,0)*min(sout[cell0], sin[cell1]) + min(f,0)*min(sin[cell0], sout[cell1])
// is formed here from the high-order residual and the scale factors of the two
// cells, by both of them alike: a pass over the edges that stored it moved 453
// MB a launch beside the 470 MB of this pass (x1.40962, six species: 105 + 95
// us, 134 us here).
template <int NE>
KB k_fct_cell2(const Instance I, float *__restrict__ out) {
  constexpr int G = HEXDYN_G_FCT_CELL2;
  const int c = wave_entity(I);
  if (c >= I.n.C) return;
  const int k = lane();
  const int L = I.n.L, NT = I.n.NT;
  const int n = I.m.neoc[c];
  int e[NE], o[NE];
#pragma unroll
  for (int s = 0; s < NE; ++s) {
    e[s] = I.m.eoc[c * NE + s];
    o[s] = I.m.ocell[c * NE + s];
  }
  SlotRow<NE> sgr = slot_row<NE>(I.m.csign + c * NE);
  const float ia = uni_load(I.m.invarea + c);
  const float rdzw = AT(I.z.rdzw, 0, k);
  const float target = AT(I.b.target, c, k);
#pragma unroll
  for (int s = 0; s < NE; ++s) {
    fence(e[s]);
    fence(o[s]);
  }
  for (int sp0 = (int)blockIdx.y * G; sp0 < NT; sp0 += (int)gridDim.y * G) {
    float hres[G][NE], sio[G][NE], soo[G][NE], si[G], so[G], vr[G], ms[G];
#pragma unroll
    for (int g = 0; g < G; ++g) {
      const int sq = clamp_sp(sp0 + g, NT);
      const int ps = sq * I.n.C;
#pragma unroll
      for (int s = 0; s < NE; ++s) {
        hres[g][s] = AT(I.b.fct_hres, sq * I.n.E + e[s], k);
        sio[g][s] = AT(I.b.fct_sin, ps + o[s], k);
        soo[g][s] = AT(I.b.fct_sout, ps + o[s], k);
      }
      si[g] = AT(I.b.fct_sin, ps + c, k);
      so[g] = AT(I.b.fct_sout, ps + c, k);
      vr[g] = AT(I.b.fct_vres, ps + c, k);
      ms[g] = AT(I.b.fct_mass, ps + c, k);
    }
    keep(hres, sio, soo, si, so, vr, ms);
    SlotRow<NE> sgs = sgr;
    settle(sgs);
    float sg[NE];
    slot_vals(sgs, sg);
#pragma unroll
    for (int g = 0; g < G; ++g) {
      if (sp0 + g >= NT) break;
      const float si_m = up1(si[g]), so_m = up1(so[g]);
      float v = vr[g];
      if (k >= 1 && k < L) v = max0(v) * pmin(so_m, si[g]) + min0(v) * pmin(so[g], si_m);
      const float v_p = dn1(v);
      float mass = ms[g];
#pragma unroll
      for (int s = 0; s < NE; ++s)
        if (s < n) {
          const bool first = sg[s] > 0.0f;  // this cell is the edge's first
          const float so1 = first ? so[g] : soo[g][s], si1 = first ? si[g] : sio[g][s];
          const float so2 = first ? soo[g][s] : so[g], si2 = first ? sio[g][s] : si[g];
          const float f = hres[g][s];
          const float lim = max0(f) * pmin(so1, si2) + min0(f) * pmin(si1, so2);
          const float sgn = -sg[s];
          mass = mass + (sgn * lim) * ia;
        }
      mass = mass - rdzw * (v_p - v);
      if (k < L) AT(out, (sp0 + g) * I.n.C + c, k) = max0(mass / target);
    }
  }
}

// q < 0 -> 0 as a where-assignment (-0.0 and NaN keep their bits); src may be dst
KB k_clamp(const Instance I, const float *src, float *dst, int rows) {
  const int r = wave_entity(I);
  if (r >= rows) return;
  const int k = lane();
  if (k >= I.n.RS) return;
  const float x = AT(src, r, k);
  AT(dst, r, k) = x < 0.0f ? 0.0f : x;
}

// Wavefronts per block of a gather kernel: the handle's launch table when the
// first kernel argument is the Instance, else 4.
template <class T>
inline int wpb_from(const char *, const T &) {
  return 4;
}
inline int wpb_from(const char *name, const Instance &I) { return I.tune ? I.tune->waves_per_block(name) : 4; }
template <class A0, class... A>
inline int launch_wpb(const char *name, const A0 &a0, const A &...) {
  return wpb_from(name, a0);
}

template <class T>
inline void set_wpb(T &, int) {}
inline void set_wpb(Instance &I, int wpb) { I.n.WPB = wpb; }

template <typename K, typename... A>
inline void launch_named(const char *name, K kernel, int n, int gy, hipStream_t s, A... args) {
  if (n <= 0 || gy <= 0) return;
  const int wpb = launch_wpb(name, args...);
  (set_wpb(args, wpb), ...);  // the launch's own copy of the Instance carries its tile
  if (g_prof_on) prof_mark(name, s, 1);
  hipLaunchKernelGGL(kernel, dim3(nblocks(n, wpb), gy), dim3(64 * wpb), 0, s, args...);
  if (g_prof_on) prof_mark(name, s, 0);
}
#define launch(kernel, ...) launch_named(#kernel, kernel, __VA_ARGS__)

// two gather passes in one launch, n0 rows of the first and n1 of the second
template <typename K, typename... A>
inline void launch_pair(const char *name, K kernel, int n0, int n1, int gy, hipStream_t s, Instance I, A... args) {
  const int wpb = wpb_from(name, I);
  I.n.WPB = wpb;
  const int nb0 = (nblocks(n0, wpb) + 7) & ~7;
  if (g_prof_on) prof_mark(name, s, 1);
  hipLaunchKernelGGL(kernel, dim3(nb0 + nblocks(n1, wpb), gy), dim3(64 * wpb), 0, s, I, nb0, args...);
  if (g_prof_on) prof_mark(name, s, 0);
}

// column kernels: W cells per block of 64*W threads
template <int W, class K, class... A>
inline void launch_col_named(const char *name, K kernel, int n, hipStream_t s, A... args) {
  if (n <= 0) return;
  if (g_prof_on) prof_mark(name, s, 1);
  hipLaunchKernelGGL(kernel, dim3((n + W - 1) / W), dim3(64 * W), 0, s, args...);
  if (g_prof_on) prof_mark(name, s, 0);
}

inline int check() {
  const hipError_t e = hipGetLastError();
  return e == hipSuccess ? 0 : -1;
}

}  // namespace

// ------------------------------------------------------------------ phases
// NE: maxEdges of the mesh (6 or 7); kernels are instantiated for both.
#define NEDISPATCH(I, call6, call7) \
  do {                              \
    if ((I).n.ME == 6) {            \
      call6;                        \
    } else {                        \
      call7;                        \
    }                               \
  } while (0)
#define LAUNCH_NE(I, kernel, ...) \
  NEDISPATCH(I, launch_named(#kernel, kernel<6>, __VA_ARGS__), launch_named(#kernel, kernel<7>, __VA_ARGS__))

// The edge-tiled flux pass runs unless the mesh has a tile with more than
// HX_TILE_U distinct stencil cells or the caller set a launch shape for the
// gather form (k_diag_edge_flux) explicitly.
inline bool tiled_flux_on(const Instance &I) {
  return I.n.TU > 0 && !(I.tune && I.tune->find("k_diag_edge_flux") >= 0);
}

// with_w: the whole step's recovery left w (and hdiv) to this pass over the
// cells; cells_done: the step's opening pass formed the cells' part
static int diagnostics(const Instance &I, int rk, int with_w, int cells_done, hipStream_t s) {
  // divergence and vorticity are read only by the horizontal mixing, from
  // the diagnostics that open a subcycle (rk 3, and the step's first), or by
  // an export between phases
  const int store_mix = rk == 3 || I.k.store_flux ? 1 : 0;
  const bool whole = with_w && I.n.VP;
  if (with_w) {
#define REC_W(NE) \
  (rk == 3 ? (whole ? RW(NE, false, true) : RW(NE, false, false)) : (whole ? RW(NE, true, true) : RW(NE, true, false)))
#define RW(NE, HD, DI) launch_named("k_rec_w", k_rec_w<NE, HD, DI>, I.n.C, 1, s, I, store_mix)
    NEDISPATCH(I, REC_W(6), REC_W(7));
#undef RW
#undef REC_W
  }
  if (whole || cells_done) {
  } else if (I.n.VP) {
    LAUNCH_NE(I, k_diag_cv, I.n.C, 1, s, I, (const float *)I.b.u, store_mix);
  } else {
    launch(k_diag_vertex, I.n.V, 1, s, I, (const float *)I.b.u, store_mix);
    LAUNCH_NE(I, k_diag_cell, I.n.C, 1, s, I, (const float *)I.b.u, store_mix);
  }
  const float *u = I.b.u;
  const bool six = I.n.ME == 6;
  if (I.k.fused && tiled_flux_on(I)) {
    const int ntiles = (I.n.E + HX_TILE_E - 1) / HX_TILE_E;
    if (g_prof_on) prof_mark("k_diag_edge_flux_t", s, 1);
    auto kt = rk == 3 ? (six ? k_diag_edge_flux_t<6, true> : k_diag_edge_flux_t<7, true>)
                      : (six ? k_diag_edge_flux_t<6, false> : k_diag_edge_flux_t<7, false>);
    hipLaunchKernelGGL(kt, dim3(ntiles), dim3(64 * HX_TILE_E), 0, s, I, u);
    if (g_prof_on) prof_mark("k_diag_edge_flux_t", s, 0);
  } else if (I.k.fused) {  // diagnostics after stage rk feed stage rk % 3 + 1 (the next subcycle's first after rk 3)
    if (rk == 3)
      launch_named("k_diag_edge_flux", six ? k_diag_edge_flux<6, true> : k_diag_edge_flux<7, true>, I.n.E, 1, s, I,
                   u);
    else
      launch_named("k_diag_edge_flux", six ? k_diag_edge_flux<6, false> : k_diag_edge_flux<7, false>, I.n.E, 1, s,
                   I, u);
  } else {
    if (rk == 3)
      launch_named("k_diag_edge", six ? k_diag_edge<6, true> : k_diag_edge<7, true>, I.n.E, 1, s, I, u);
    else
      launch_named("k_diag_edge", six ? k_diag_edge<6, false> : k_diag_edge<7, false>, I.n.E, 1, s, I, u);
  }
  return check();
}

int solve_diagnostics(const Instance &I, int rk, int with_w, hipStream_t s) {
  return diagnostics(I, rk, with_w, 0, s);
}

int begin_step(const Instance &I, hipStream_t s) {
  if (I.n.NM > 0) {
#define BEGIN(NE, DI) launch_pair("k_begin", k_begin<NE, DI>, I.n.E, I.n.C, 1, s, I)
    NEDISPATCH(I, I.n.VP ? BEGIN(6, true) : BEGIN(6, false), I.n.VP ? BEGIN(7, true) : BEGIN(7, false));
#undef BEGIN
  }
  return diagnostics(I, 3, 0, I.n.NM > 0 && I.n.VP, s);
}

int begin_subcycle(const Instance &I, int sub, hipStream_t s) {
  (void)sub;
  if (!I.k.fused)  // the whole step forms the implicit coefficients in the stages' column passes
    launch_col_named<COLW_VC>("k_vcoef", k_vcoef, I.n.C, s, I, I.k.dts[0], (const float *)I.b.s_exner,
                              (const float *)I.b.s_theta, (const float *)I.b.s_rtheta_p);
  // with mixing, kdiff rides on the cell pass and the del2 u increment on the
  // edge pass (the pool is written once)
  if (I.k.mixing) {
    if (I.n.NM > 0)
      NEDISPATCH(I, launch_named("k_sub_cell", k_sub_cell<6, true, true>, I.n.C, 1, s, I),
                 launch_named("k_sub_cell", k_sub_cell<7, true, true>, I.n.C, 1, s, I));
    else
      NEDISPATCH(I, launch_named("k_sub_cell", k_sub_cell<6, true, false>, I.n.C, 1, s, I),
                 launch_named("k_sub_cell", k_sub_cell<7, true, false>, I.n.C, 1, s, I));
    launch_named("k_sub_edge", k_sub_edge<true>, I.n.E, 1, s, I);
  } else {
    if (I.n.NM > 0)
      NEDISPATCH(I, launch_named("k_sub_cell", k_sub_cell<6, false, true>, I.n.C, 1, s, I),
                 launch_named("k_sub_cell", k_sub_cell<7, false, true>, I.n.C, 1, s, I));
    else
      NEDISPATCH(I, launch_named("k_sub_cell", k_sub_cell<6, false, false>, I.n.C, 1, s, I),
                 launch_named("k_sub_cell", k_sub_cell<7, false, false>, I.n.C, 1, s, I));
    launch_named("k_sub_edge", k_sub_edge<false>, I.n.E, 1, s, I);
  }
  if (I.k.mixing) {
    const bool mix4 = I.k.mix4 != 0, lap = mix4 && I.n.VP;
    if (mix4 && !lap) {
      LAUNCH_NE(I, k_mix_lapdiv, I.n.C, 1, s, I);
      launch(k_mix_lapvort, I.n.V, 1, s, I);
    }
#define MIX(NE, M4, LA) launch_named("k_mix_cell", k_mix_cell<NE, M4, LA>, I.n.C, 1, s, I)
#define MIX_NE(NE) (lap ? MIX(NE, true, true) : mix4 ? MIX(NE, true, false) : MIX(NE, false, false))
    NEDISPATCH(I, MIX_NE(6), MIX_NE(7));
#undef MIX_NE
#undef MIX
    if (mix4)
      NEDISPATCH(I, launch_pair("k_mix4", k_mix4<6>, I.n.E, I.n.C, 1, s, I),
                 launch_pair("k_mix4", k_mix4<7>, I.n.E, I.n.C, 1, s, I));
  }
  return check();
}

// the column pass of a stage on the whole-step path
template <int NE>
void stage_columns(const Instance &I, int stage, int sub, hipStream_t s) {
  const int n = I.k.steps[stage - 1];
  const float dts = I.k.dts[stage - 1];
  const bool order3 = I.k.order == 3, vc = stage == 1 || (stage == 2 && order3);
  const bool corr = stage > 1, mix = I.k.mixing != 0, last = n == 1;
  // a later substep's damping reads rtheta_pp_old; with two substeps the
  // second takes the zero without a store and a reload
  const int store_old = n > 2 ? 1 : 0;
  // stage 1 of the third-order scheme is one substep, and stage 2 forms its own coefficients
  const int store_cof = !(stage == 1 && order3 && last) ? 1 : 0;
  const int closing = stage == 3 && sub == I.k.splits ? 1 : 0;  // the working fields the step leaves current
  const int store_t = !last || closing ? 1 : 0;
  const RecArgs ra{sub, I.k.inv_steps[stage - 1], stage == 3 || (stage == 1 && order3) ? 1 : 0, closing};
#define COL(VCV, CO, MX, LA, S3V)                                                                                \
  launch_col_named<COLW_AC>("k_col", k_col<NE, VCV, CO, MX, LA, S3V>, I.n.C, s, I, dts,                          \
                            (const float *)I.b.rtheta_p, store_old, store_cof, store_t, ra)
#define COL_MIX(VCV, CO, LA, S3V) (mix ? COL(VCV, CO, true, LA, S3V) : COL(VCV, CO, false, LA, S3V))
  if (stage == 3) {
    last ? COL_MIX(false, true, true, true) : COL_MIX(false, true, false, false);
  } else if (vc) {
    corr ? (last ? COL_MIX(true, true, true, false) : COL_MIX(true, true, false, false))
         : (last ? COL_MIX(true, false, true, false) : COL_MIX(true, false, false, false));
  } else {
    last ? COL_MIX(false, true, true, false) : COL_MIX(false, true, false, false);
  }
#undef COL_MIX
#undef COL
}

int dyn_tend(const Instance &I, int stage, int sub, hipStream_t s) {
  if (I.k.fused) {
    // the edge fluxes came with the preceding diagnostics
    const int store_avg = I.k.steps[stage - 1] > 2 ? 1 : 0, store_rup = I.k.steps[stage - 1] > 1 || stage == 3 ? 1 : 0;
#define MOM(NE, RW) \
  launch_named("k_tend_mom_ac", k_tend_mom_ac<NE, RW>, I.n.E, 1, s, I, I.k.dts[stage - 1], store_avg, store_rup)
    if (I.n.REFW)
      NEDISPATCH(I, MOM(6, true), MOM(7, true));
    else
      NEDISPATCH(I, MOM(6, false), MOM(7, false));
#undef MOM
    NEDISPATCH(I, stage_columns<6>(I, stage, sub, s), stage_columns<7>(I, stage, sub, s));
    return check();
  }
  if (stage == 2 && I.k.order == 3)
    launch_col_named<COLW_VC>("k_vcoef", k_vcoef, I.n.C, s, I, I.k.dts[1], (const float *)I.b.s_exner,
                              (const float *)I.b.theta, (const float *)I.b.rtheta_p);
  if (I.n.REFW)
    NEDISPATCH(I, launch_named("k_tend_mom", k_tend_mom<6, true>, I.n.E, 1, s, I),
               launch_named("k_tend_mom", k_tend_mom<7, true>, I.n.E, 1, s, I));
  else
    NEDISPATCH(I, launch_named("k_tend_mom", k_tend_mom<6, false>, I.n.E, 1, s, I),
               launch_named("k_tend_mom", k_tend_mom<7, false>, I.n.E, 1, s, I));
  if (stage > 1)
    NEDISPATCH(I, launch_named("k_tend_flux", k_tend_flux<6, true>, I.n.E, 1, s, I),
               launch_named("k_tend_flux", k_tend_flux<7, true>, I.n.E, 1, s, I));
  else
    NEDISPATCH(I, launch_named("k_tend_flux", k_tend_flux<6, false>, I.n.E, 1, s, I),
               launch_named("k_tend_flux", k_tend_flux<7, false>, I.n.E, 1, s, I));
  {
    const bool corr = stage > 1, mix = I.k.mixing != 0;
#define TEND_CELL(NE, CO, MX) launch_named("k_tend_cell", k_tend_cell<NE, CO, MX>, I.n.C, 1, s, I)
#define TEND_CELL_NE(NE)                           \
  (corr ? (mix ? TEND_CELL(NE, true, true) : TEND_CELL(NE, true, false)) \
        : (mix ? TEND_CELL(NE, false, true) : TEND_CELL(NE, false, false)))
    NEDISPATCH(I, TEND_CELL_NE(6), TEND_CELL_NE(7));
#undef TEND_CELL_NE
#undef TEND_CELL
  }
  return check();
}

template <int NE>
void substep_columns(const Instance &I, int stage, int ss, int sub, hipStream_t s) {
  const float dts = I.k.dts[stage - 1];
  const bool last = I.k.fused && ss == I.k.steps[stage - 1];
  const RecArgs ra{sub, I.k.inv_steps[stage - 1], stage == 3 || (stage == 1 && I.k.order == 3) ? 1 : 0,
                   stage == 3 && sub == I.k.splits ? 1 : 0};
#define AC(FI, LA, S3V) launch_col_named<COLW_AC>("k_ac_cell", k_ac_cell<NE, FI, LA, S3V>, I.n.C, s, I, dts, 1, ra)
  if (ss == 1)
    AC(true, false, false);
  else if (!last)
    AC(false, false, false);
  else if (stage == 3)
    AC(false, true, true);
  else
    AC(false, true, false);
#undef AC
}

int acoustic_substep(const Instance &I, int stage, int ss, int sub, int damp_prev, hipStream_t s) {
  const float dts = I.k.dts[stage - 1];
  const int n = I.k.steps[stage - 1];
  // fused: the first edge update ran with the momentum tendency, the first column update with the tendencies
  if (I.k.fused && ss == 1) return check();
  const float coef = I.k.dts_inv_coef[stage - 1];
  const bool avgrp = I.k.fused && n == 2;
  if (ss == 1)
    launch_named("k_ac_edge", k_ac_edge<true, false, false>, I.n.E, 1, s, I, dts, coef);
  else if (damp_prev && avgrp)
    launch_named("k_ac_edge", k_ac_edge<false, true, true>, I.n.E, 1, s, I, dts, coef);
  else if (damp_prev)
    launch_named("k_ac_edge", k_ac_edge<false, true, false>, I.n.E, 1, s, I, dts, coef);
  else if (avgrp)
    launch_named("k_ac_edge", k_ac_edge<false, false, true>, I.n.E, 1, s, I, dts, coef);
  else
    launch_named("k_ac_edge", k_ac_edge<false, false, false>, I.n.E, 1, s, I, dts, coef);
  NEDISPATCH(I, substep_columns<6>(I, stage, ss, sub, s), substep_columns<7>(I, stage, ss, sub, s));
  return check();
}

int divergence_damping(const Instance &I, int stage, hipStream_t s) {
  launch(k_divdamp, I.n.E, 1, s, I, I.k.dts_inv_coef[stage - 1]);
  return check();
}

template <bool S3>
void recover_edges(const Instance &I, int sub, float inv, bool damp, bool avgrp, float coef, float dts,
                   hipStream_t s) {
#define REC(DA, AV, RH) launch_named("k_rec_edge", k_rec_edge<S3, DA, AV, RH>, I.n.E, 1, s, I, sub, inv, coef, dts)
  if (I.k.fused)
    damp ? (avgrp ? REC(true, true, true) : REC(true, false, true))
         : (avgrp ? REC(false, true, true) : REC(false, false, true));
  else
    REC(false, false, false);  // the phase entry points damp in a pass of their own and keep ru_avg
#undef REC
}

// w_later: the transport's first pass recovers the last stage's w
int recover(const Instance &I, int stage, int sub, int damp, int w_later, hipStream_t s) {
  const bool last = stage == 3 && sub == I.k.splits;
  const float inv = I.k.inv_steps[stage - 1];
  const bool avgrp = I.k.fused && I.k.steps[stage - 1] == 1;
  const float coef = I.k.dts_inv_coef[stage - 1];
  if (stage == 3)
    recover_edges<true>(I, sub, inv, damp != 0, avgrp, coef, I.k.dts[stage - 1], s);
  else
    recover_edges<false>(I, sub, inv, damp != 0, avgrp, coef, I.k.dts[stage - 1], s);
  if (I.k.fused) {
    // the column pass recovered the rest; w and hdiv come with the diagnostics
    // that follow, except after a step's last stage, which has none
    if (last && !w_later)
      NEDISPATCH(I, launch_named("k_rec_w", k_rec_w<6, false, false>, I.n.C, 1, s, I, 0),
                 launch_named("k_rec_w", k_rec_w<7, false, false>, I.n.C, 1, s, I, 0));
  } else if (stage == 3) {
    NEDISPATCH(I, launch_named("k_rec_cell", k_rec_cell<6, true>, I.n.C, 1, s, I, sub, inv),
               launch_named("k_rec_cell", k_rec_cell<7, true>, I.n.C, 1, s, I, sub, inv));
  } else {
    NEDISPATCH(I, launch_named("k_rec_cell", k_rec_cell<6, false>, I.n.C, 1, s, I, sub, inv),
               launch_named("k_rec_cell", k_rec_cell<7, false>, I.n.C, 1, s, I, sub, inv));
  }
  return check();
}

// Grid rows of a scalar pass over n entities in batches of g species: a row a
// batch where the launch stays small (HX_SMALL), so that the batches run side by
// side instead of one memory round trip after another: a step with six species
// 280 -> 266 us at x1.162, 341 -> 332 at x1.642, 470 -> 465 at x1.2562 (there the
// cell passes alone).  Above, the batches fill the chip as well one after the other
// and share the species-independent rows: 1177 us at x1.10242, 1183 with a row a
// batch.
inline int species_rows(const Instance &I, int n, int g) {
  const int batches = (I.n.NT + g - 1) / g;
  return batches > 1 && (long long)n * batches <= HX_SMALL ? batches : 1;  // without species a launch of one row
}

int scalars_stage(const Instance &I, int stage, int with_w, hipStream_t s) {
  const float dt = I.k.sca_dt[stage - 1];
  const float *qin = stage == 1 ? I.b.q : I.b.q_stage;  // stage 1 starts from the published scalars
  if (stage < 3 || !I.k.monotonic) {
    const int rows = species_rows(I, I.n.E, HEXDYN_G_SC_EDGE);
    if (with_w)
      NEDISPATCH(I, launch_pair("k_sc_edge_w", k_sc_edge_w<6>, I.n.E, I.n.C, rows, s, I, qin, I.b.ev),
                 launch_pair("k_sc_edge_w", k_sc_edge_w<7>, I.n.E, I.n.C, rows, s, I, qin, I.b.ev));
    else
      LAUNCH_NE(I, k_sc_edge, I.n.E, rows, s, I, qin, I.b.ev);
    LAUNCH_NE(I, k_sc_cell, I.n.C, species_rows(I, I.n.C, HEXDYN_G_SC_CELL), s, I, qin, (const float *)I.b.ev,
              I.b.q_next, dt,
              I.k.wn[stage - 1], (const float *)(I.k.physics_q ? I.b.phys_q : nullptr));
    return check();
  }
  // the limiter's old mixing ratio: the published one plus +0, or the one
  // the held scalar tendency moved (x + -0 == x keeps its bits)
  const float *qold = I.b.q;
  float qadd = 0.0f;
  if (I.k.physics_q) {
    launch(k_fct_source, I.n.C, 1, s, I, dt);
    qold = I.b.q_src;
    qadd = -0.0f;
  }
  LAUNCH_NE(I, k_fct_edge1, I.n.E, species_rows(I, I.n.E, HEXDYN_G_FCT_EDGE1), s, I, qin, dt, qold, qadd);
  {
    const int rows = species_rows(I, I.n.C, HEXDYN_G_FCT_CELL1);
#define FCT1(NE, PAIR) launch_named("k_fct_cell1", k_fct_cell1<NE, PAIR>, I.n.C, rows, s, I, qin, dt, qold, qadd)
    if (I.n.OCP)
      NEDISPATCH(I, FCT1(6, true), FCT1(7, true));
    else
      NEDISPATCH(I, FCT1(6, false), FCT1(7, false));
#undef FCT1
  }
  LAUNCH_NE(I, k_fct_cell2, I.n.C, species_rows(I, I.n.C, HEXDYN_G_FCT_CELL2), s, I, I.b.q_next);
  return check();
}

int rebuild_saved(const Instance &I, hipStream_t s) {
  LAUNCH_NE(I, k_rebuild_cell, I.n.C, 1, s, I);
  launch(k_rebuild_edge, I.n.E, 1, s, I);
  return check();
}

int rebuild_cells(const Instance &I, hipStream_t s) {
  LAUNCH_NE(I, k_rebuild_cell, I.n.C, 1, s, I);
  return check();
}

int clamp_scalars(const Instance &I, const float *src, float *dst, hipStream_t s) {
  launch(k_clamp, I.n.NT * I.n.C, 1, s, I, src, dst, I.n.NT * I.n.C);
  return check();
}

}  // namespace HEXDYN_NS
}  // namespace hexdyn
