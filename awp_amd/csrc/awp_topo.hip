// Curvilinear topography: the velocity and stress (with coarse-grained Q)
// updates on a grid z = g(r) f(x, y) that follows the free surface, and the
// builders of the metric arrays f*, g*.
//
//   topo_velocity_interior_H  dtopo_vel_111 (levels 3 <= k < nz-6) and
//                             dtopo_vel_112 (top six levels), reference
//                             src/topography/velocity.cu:28-268,
//                             kernels/velocity_unroll.cu, optimized_velocity.cu:1040-1627
//   topo_stress_interior_H    dtopo_str_111 / dtopo_str_112,
//                             src/topography/stress_attenuation.cu:25-130,
//                             kernels/stress_attenuation.cu:74-1410
//   awp_topo_metrics_f/_g     metrics_build_f/_g, metrics/metrics.c:35-41,
//                             223-229 with metrics/kernel.c:3-292
//   awp_topo_geom_custom      geom_custom, geometry/geometry.c:188-210
//
// Lane map: one lane per level k (64 consecutive levels per wave, so every
// field access of a wave is one contiguous 256-byte run); the waves of a
// workgroup share one column chunk in LDS and march along i (topo_rates_kernel
// <ST, 1> along j).  The top six levels' one-sided rows are per-lane
// coefficients of the wave at the surface, in the same launch.
// Every expression keeps the reference's operand order and literal types
// (double where it writes double literals), so results match the CPU
// oracle bit for bit.
#include "awp_common.h"
#include "awp_math.h"
#include "awp_store.h"
#include "awp_topo_coef.h"
#include "awp_tuning.h"
#include "../../include/awp_hip.h"

namespace {

// float tables, as the reference's `const float` initialisers compute them
template <int R, int C>
struct FTab {
  float v[R][C];
};
template <int R, int C>
constexpr FTab<R, C> ftab(const double (&a)[R][C]) {
  FTab<R, C> t{};
  for (int r = 0; r < R; ++r)
    for (int c = 0; c < C; ++c) t.v[r][c] = (float)a[r][c];
  return t;
}

__constant__ FTab<6, 9> c_str_phdz4r = ftab(TS_PHDZ4R);
__constant__ FTab<6, 7> c_str_dz4r = ftab(TS_DZ4R);
__constant__ FTab<6, 8> c_str_dhz4r = ftab(TS_DHZ4R);
__constant__ FTab<6, 9> c_str_pdhz4r = ftab(TS_PDHZ4R);

#define P4F(q) ((float)TOPO_P4[q])
#define D4F(q) ((float)TOPO_D4[q])

// Geometry of one grid: wavefield strides (32-bit: checked on the host) and
// the metric row length.
struct TGeom {
  int nx, ny, nz;
  int yl, sl, frow;
  int bi, bj, ei, ej;  // bounds of the launch (topographic for velocity,
                       // array indices for stress)
};

template <class ST>
struct TField {
  const typename ST::T* p;
  float s;
  __device__ __forceinline__ float operator[](int idx) const { return ST::ld(p, idx, s); }
};

struct TMetrics {
  const float *f, *f_1, *f_2, *f_c, *f1_1, *f1_2, *f1_c, *f2_1, *f2_2, *f2_c;
  const float *g, *g3, *g3_c, *g_c;
};

template <class ST>
struct TopoVelArgs {
  typename ST::T *u1, *u2, *u3;
  TField<ST> s11, s12, s13, s22, s23, s33;
  const float *rho, *dcrjx, *dcrjy, *dcrjz;
  TMetrics M;
  float iu1, iu2, iu3, su1, su2, su3;  // velocity scales (decode / encode)
  float a, nu;
};

// Orders one wave's LDS stores before its lanes read each other's values
// (release, then acquire, at wavefront scope).  Enough where a wave reads
// only the LDS it writes itself; a chunk of several waves sharing LDS needs
// the workgroup barrier.
__device__ __forceinline__ void wave_lds_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// ---------------------------------------------------------------------------
// Velocity: dtopo_vel_111_unroll (velocity_unroll.cu:1-461) on levels
// 3 <= k < nz-6 and dtopo_vel_112 (optimized_velocity.cu:1040-1627) on the top
// six, in one kernel.
//
// A workgroup owns a chunk of 64 * nseg levels of one j row (several rows of
// one-wave chunks) and marches along i.  At every plane each lane forms, at
// its own level, the horizontal 4-point interpolants whose z derivatives the
// metric terms need, and publishes them (with its own s13, s23, s33) in LDS;
// the 7-point (9-point on the top rows) z sums then read the neighbouring
// levels from LDS.  The x neighbours travel in register windows.  A chunk
// writes all but its 3 outermost levels on either side, so chunks overlap by
// six; the last one ends at level nz-1 and takes the one-sided top rows (table
// row kk = nz-1-k) too: its waves that hold any form every z sum with
// per-lane coefficients, so their lanes do not diverge.
#define VT_MAXW 8    // waves per workgroup at most
#define VT_NL 9      // staged LDS columns per row
#define VT_PAD 4     // LDS floats before and after a staged column: the halo lanes of
                     // a chunk read up to 3 levels outside it and discard the sums

// The k tiling of a curvilinear launch (topo_tiles): chunks of nseg waves that
// share one LDS column.
struct VelTiles {
  int nint;   // interior chunks (ch - 6 outputs each, from level 3)
  int ktop0;  // first level of the top chunk (nz - ch, may be negative)
  int wtop0;  // first level the top chunk writes
  int ichunk; // planes per march
  int njt;    // j tiles (velocity)
  int nseg;   // waves per chunk (64 levels each)
  int ch;     // levels per chunk, 64 * nseg
  int step;   // ch - 6
  int rj;     // j rows per workgroup (nseg * rj waves)
  int wsync;  // 1: a wave that reads only its own LDS syncs at wave scope, not the workgroup's
};

// A float read at a wave-uniform index of an array that no kernel in flight
// writes: through the constant address space it is a scalar load.
typedef const __attribute__((address_space(4))) float* uniform_ptr;
__device__ __forceinline__ float uld(const float* a, int i) { return ((uniform_ptr)a)[i]; }

// Order of an interior 7-point row: the middle, then from one end.
__host__ __device__ constexpr int rt_mid(int t) { return t == 0 ? 3 : t <= 3 ? t - 1 : t; }

// Per-lane coefficients [term][class] of the waves with one-sided rows: class
// 0..5 is the row of level nz-1-class, the level furthest from the top
// first; class 6 the interior row in its own order, then zeros for the terms
// a one-sided row has more (they weigh the lane's own level).
#define VT_ZC 0    // dhpz4 (times g_c)
#define VT_ZN 9    // dphz4 (times g)
#define VT_DHZ 18  // dhz4
#define VT_DZ 26   // dz4
#define VT_N 33
struct VelTop {
  float v[VT_N][8];
};
constexpr VelTop vel_top() {
  VelTop T{};
  constexpr int dho[4] = {2, 0, 1, 3}, dzo[4] = {1, 0, 2, 3};
  for (int c = 0; c < 6; ++c) {
    for (int t = 0; t < 9; ++t) {
      T.v[VT_ZC + t][c] = (float)TV_DHPZ4R[c][8 - t];
      T.v[VT_ZN + t][c] = (float)TV_DPHZ4R[c][8 - t];
    }
    for (int t = 0; t < 8; ++t) T.v[VT_DHZ + t][c] = (float)TV_DHZ4R[c][7 - t];
    for (int t = 0; t < 7; ++t) T.v[VT_DZ + t][c] = (float)TV_DZ4R[c][6 - t];
  }
  for (int t = 0; t < 7; ++t) {
    T.v[VT_ZC + t][6] = (float)TV_DHPZ4[rt_mid(t)];
    T.v[VT_ZN + t][6] = (float)TV_DPHZ4[rt_mid(t)];
  }
  for (int t = 0; t < 4; ++t) {
    T.v[VT_DHZ + t][6] = (float)TOPO_D4[dho[t]];
    T.v[VT_DZ + t][6] = (float)TOPO_D4[dzo[t]];
  }
  return T;
}
__constant__ VelTop c_vel_top = vel_top();

// All three components in one launch: it reads 10 arrays and writes 3 where a
// launch per component reads 15 (384x384x192: 500 against 530 us; 256x256x192
// 233 against 243).
template <class ST>
__global__ __launch_bounds__(64 * VT_MAXW) void topo_vel_kernel(const TopoVelArgs<ST> A,
                                                               const TGeom G,
                                                               const VelTiles V) {
  constexpr int NL = VT_NL;
  constexpr int CU = 0, CV = 3, CW = 6;  // columns: two interpolants and a stress each
  extern __shared__ float vt_lds[];  // [parity][row][column][VT_PAD + ch + VT_PAD]
  __shared__ float s_top[VT_N * 8];
  const int lane = (int)threadIdx.x;
  const int w = (int)threadIdx.y;
  const int seg = w % V.nseg, row = w / V.nseg;
  // k chunks fastest, then j tiles, then i chunks, a contiguous run of them
  // per XCD: the rows that neighbouring j tiles share meet in one L2
  const int b = awp_xcd_remap((int)blockIdx.x, (int)gridDim.x);
  const int t = b % (V.nint + 1), jt = b / (V.nint + 1) % V.njt;
  const int ic = b / ((V.nint + 1) * V.njt);
  const bool top = t == V.nint;
  if (top) {  // uniform over the workgroup
    for (int e = w * 64 + lane; e < VT_N * 8; e += V.nseg * V.rj * 64)
      s_top[e] = (&c_vel_top.v[0][0])[e];
    __syncthreads();
  }
  const int k0 = top ? V.ktop0 : V.step * t;
  const int kl = seg * 64 + lane;  // level within the chunk
  const int k = k0 + kl;
  const int nz = G.nz;
  // levels this lane writes
  const int w0 = top ? V.wtop0 : V.step * t + 3;
  const int w1 = top ? nz : (V.step * t + V.ch - 3 < V.wtop0 ? V.step * t + V.ch - 3 : V.wtop0);
  const bool bnd = k >= nz - 6;  // one-sided rows (top chunk only)
  const bool topw = top && __builtin_amdgcn_readfirstlane(k0 + seg * 64 + 63) >= nz - 6;
  // every wave of the workgroup runs the same planes (uniform barrier count);
  // a wave past the last column works on a copy of it and stores nothing
  const int jw = G.bj + jt * V.rj + row;
  const bool jok = jw < G.ej;
  const int j = __builtin_amdgcn_readfirstlane(jok ? jw : G.ej - 1);
  const int ib = ic * V.ichunk;
  const int ie = ib + V.ichunk < G.ei ? ib + V.ichunk : G.ei;
  if (ib >= ie) return;  // uniform over the workgroup
  const bool out = k >= w0 && k < w1 && jok;
  const int sl = G.sl, yl = G.yl, fr = G.frow;
  // every lane reads at its own level; the top chunk of a grid with
  // nz < ch starts below level 0, and those lanes (never outputs, never read
  // by an output's stencil) read level 0 instead
  const int kr = k < 0 ? 0 : k;
  const int kg = kr + AWP_ALIGN;
  const int col0 = yl * (j + AWP_NGSL + 2) + AWP_ALIGN;   // level 0 of column (i = -10)
  const TMetrics& M = A.M;
  const int cp = V.ch + 2 * VT_PAD;
  const int own = VT_PAD + kl;          // this lane's level in a staged column
  const int lb = VT_PAD + nz - 1 - k0;  // level nz-1 (top chunk)
  const int cls = bnd ? nz - 1 - k : 6;

  // per-level weights of the z sums, term by term in the order they are added
  // (7 terms; 9 in the waves with one-sided rows)
  float cz[9], czp[9];
  if (!topw) {
#pragma unroll
    for (int m = 0; m < 7; ++m) {
      const int kk2 = kg + rt_mid(m) - 3;  // >= align - 3
      cz[m] = (float)TV_DHPZ4[rt_mid(m)] * M.g_c[kk2];
      czp[m] = (float)TV_DPHZ4[rt_mid(m)] * M.g[kk2];
    }
  } else {
#pragma unroll
    for (int m = 0; m < 9; ++m) {
      const int kk2 = AWP_ALIGN + (bnd ? nz - 9 + m : kr + (m < 7 ? rt_mid(m) - 3 : 0));
      cz[m] = s_top[(VT_ZC + m) * 8 + cls] * M.g_c[kk2];
      czp[m] = s_top[(VT_ZN + m) * 8 + cls] * M.g[kk2];
    }
  }
  // z sum of a staged column with weights c
  auto zsum = [&](const float(&c)[9], const float* L) {
    float acc = 0.f;
    if (!topw) {
#pragma unroll
      for (int m = 0; m < 7; ++m) {
        const float x = c[m] * L[own + rt_mid(m) - 3];
        acc = m == 0 ? x : acc + x;
      }
    } else {
#pragma unroll
      for (int m = 0; m < 9; ++m) {
        const float x = c[m] * L[bnd ? lb - 8 + m : own + (m < 7 ? rt_mid(m) - 3 : 0)];
        acc = m == 0 ? x : acc + x;
      }
    }
    return acc;
  };
  // acc (if any) plus the terms of dhz4 / dz4 on a staged column
  auto add_dhz = [&](bool first, float acc, const float* L) {
    if (!topw) {
      const float x = D4F(2) * L[own];
      acc = first ? x : acc + x;
      acc = acc + D4F(0) * L[own - 2];
      acc = acc + D4F(1) * L[own - 1];
      return acc + D4F(3) * L[own + 1];
    }
#pragma unroll
    for (int m = 0; m < 8; ++m) {
      const int o = m == 1 ? -2 : m == 2 ? -1 : m == 3 ? 1 : 0;
      const float x = s_top[(VT_DHZ + m) * 8 + cls] * L[bnd ? lb - 7 + m : own + o];
      acc = first && m == 0 ? x : acc + x;
    }
    return acc;
  };
  auto add_dz = [&](float acc, const float* L) {
    if (!topw) {
      acc = acc + D4F(1) * L[own];
      acc = acc + D4F(0) * L[own - 1];
      acc = acc + D4F(2) * L[own + 1];
      return acc + D4F(3) * L[own + 2];
    }
#pragma unroll
    for (int m = 0; m < 7; ++m) {
      const int o = m == 1 ? -1 : m == 2 ? 1 : m == 3 ? 2 : 0;
      acc = acc + s_top[(VT_DZ + m) * 8 + cls] * L[bnd ? lb - 6 + m : own + o];
    }
    return acc;
  };
  const float g3c = M.g3_c[kg], g3v = M.g3[kg];
  const float dcz = A.dcrjz[kg];
  const float dcy = uld(A.dcrjy, j + AWP_NGSL + 2);

  // x windows at level k: s11(i-2..i+1), s12(i-1..i+2), s13(i-1..i+2)
  auto P = [&](int i) { return col0 + sl * (i + AWP_NGSL + 2) + kr; };
  float s11w[4], s12x[4], s13x[4];
#pragma unroll
  for (int q = 0; q < 3; ++q) {
    s11w[q + 1] = A.s11[P(ib - 2 + q)];
    s12x[q + 1] = A.s12[P(ib - 1 + q)];
    s13x[q + 1] = A.s13[P(ib - 1 + q)];
  }
  // density at plane i-1: (j, k-1), (j, k), (j-1, k)
  float rm_k1 = A.rho[P(ib - 1) - 1], rm_k = A.rho[P(ib - 1)], rm_j = A.rho[P(ib - 1) - yl];

  for (int i = ib; i < ie; ++i) {
    const int par = i & 1;
    const int p = P(i);
#pragma unroll
    for (int q = 0; q < 3; ++q) {
      s11w[q] = s11w[q + 1];
      s12x[q] = s12x[q + 1];
      s13x[q] = s13x[q + 1];
    }
    s11w[3] = A.s11[p + sl];
    s12x[3] = A.s12[p + 2 * sl];
    s13x[3] = A.s13[p + 2 * sl];
    const float s12m2 = A.s12[p - 2 * yl], s12m1 = A.s12[p - yl], s12p1 = A.s12[p + yl];
    const float s22m1 = A.s22[p - yl], s22o = A.s22[p], s22p1 = A.s22[p + yl],
                s22p2 = A.s22[p + 2 * yl];
    const float s23m2 = A.s23[p - 2 * yl], s23m1 = A.s23[p - yl], s23o = A.s23[p],
                s23p1 = A.s23[p + yl];
    const float s12o = s12x[1], s13o = s13x[1];
    float* L = vt_lds + (par * V.rj + row) * NL * cp;
    // interpolants at this level, operands in the reference's order
    L[CU * cp + own] =
        P4F(2) * s11w[2] + P4F(0) * s11w[0] + P4F(1) * s11w[1] + P4F(3) * s11w[3];
    L[(CU + 1) * cp + own] =
        P4F(2) * s12o + P4F(0) * s12m2 + P4F(1) * s12m1 + P4F(3) * s12p1;
    L[(CU + 2) * cp + own] = s13o;
    L[CV * cp + own] =
        P4F(1) * s12x[1] + P4F(0) * s12x[0] + P4F(2) * s12x[2] + P4F(3) * s12x[3];
    L[(CV + 1) * cp + own] =
        P4F(1) * s22o + P4F(0) * s22m1 + P4F(2) * s22p1 + P4F(3) * s22p2;
    L[(CV + 2) * cp + own] = s23o;
    L[CW * cp + own] =
        P4F(1) * s13x[1] + P4F(0) * s13x[0] + P4F(2) * s13x[2] + P4F(3) * s13x[3];
    L[(CW + 1) * cp + own] =
        P4F(2) * s23o + P4F(0) * s23m2 + P4F(1) * s23m1 + P4F(3) * s23p1;
    L[(CW + 2) * cp + own] = A.s33[p];
    // density at plane i, and the velocities before the step
    const float r_k1 = A.rho[p - 1], r_k = A.rho[p], r_j = A.rho[p - yl],
                r_jk1 = A.rho[p - yl - 1];
    const float u = ST::ld(A.u1, p, A.su1), v = ST::ld(A.u2, p, A.su2),
                x = ST::ld(A.u3, p, A.su3);
    // one-wave chunks read only their own LDS rows: with wsync the waves of
    // the workgroup do not wait for each other
    if (V.wsync && V.nseg == 1)
      wave_lds_sync();
    else
      __syncthreads();

    const int q = (j + AWP_ALIGN + AWP_NGSL + 2) + (i + AWP_NGSL + 2) * fr;
    // the top rows' means are binary64 sums rounded to binary32: the sum of
    // two binary32 values rounds the same through binary64 (awp_quot's
    // theorem), and a quarter of it is exact, so one form serves every row
    const float c = 0.25f;
    const float f_dcrj = uld(A.dcrjx, i + AWP_NGSL + 2) * dcy * dcz;
    float s;
    // u1
    {
      const float rho1 = c * (r_k1 + r_jk1) + c * (r_k + r_j);
      const float Ai1 = awp_div(A.nu, uld(M.f_1, q) * g3c * rho1);
      const float z11 = zsum(cz, L + CU * cp), z12 = zsum(cz, L + (CU + 1) * cp);
      s = D4F(2) * uld(M.f_c, q) * g3c * s11w[2];
      s = s + D4F(0) * uld(M.f_c, q - 2 * fr) * g3c * s11w[0];
      s = s + D4F(1) * uld(M.f_c, q - fr) * g3c * s11w[1];
      s = s + D4F(3) * uld(M.f_c, q + fr) * g3c * s11w[3];
      s = s + D4F(2) * uld(M.f, q) * g3c * s12o;
      s = s + D4F(0) * uld(M.f, q - 2) * g3c * s12m2;
      s = s + D4F(1) * uld(M.f, q - 1) * g3c * s12m1;
      s = s + D4F(3) * uld(M.f, q + 1) * g3c * s12p1;
      s = add_dhz(false, s, L + (CU + 2) * cp);
      s = s - uld(M.f1_1, q) * z11;
      s = s - uld(M.f2_1, q) * z12;
      if (out) ST::st(A.u1, p, (A.a * u + Ai1 * s) * f_dcrj, A.iu1);
    }
    // u2
    {
      const float rho2 = c * (r_k1 + rm_k1) + c * (r_k + rm_k);
      const float Ai2 = awp_div(A.nu, uld(M.f_2, q) * g3c * rho2);
      const float z12x = zsum(cz, L + CV * cp), z22 = zsum(cz, L + (CV + 1) * cp);
      s = add_dhz(true, 0.f, L + (CV + 2) * cp);
      s = s + D4F(1) * uld(M.f, q) * g3c * s12x[1];
      s = s + D4F(0) * uld(M.f, q - fr) * g3c * s12x[0];
      s = s + D4F(2) * uld(M.f, q + fr) * g3c * s12x[2];
      s = s + D4F(3) * uld(M.f, q + 2 * fr) * g3c * s12x[3];
      s = s + D4F(1) * uld(M.f_c, q) * g3c * s22o;
      s = s + D4F(0) * uld(M.f_c, q - 1) * g3c * s22m1;
      s = s + D4F(2) * uld(M.f_c, q + 1) * g3c * s22p1;
      s = s + D4F(3) * uld(M.f_c, q + 2) * g3c * s22p2;
      s = s - uld(M.f1_2, q) * z12x;
      s = s - uld(M.f2_2, q) * z22;
      if (out) ST::st(A.u2, p, (A.a * v + Ai2 * s) * f_dcrj, A.iu2);
    }
    // u3
    {
      const float rho3 = c * (r_k + rm_k) + c * (r_j + rm_j);
      const float Ai3 = awp_div(A.nu, uld(M.f_c, q) * g3v * rho3);
      const float z13 = zsum(czp, L + CW * cp), z23 = zsum(czp, L + (CW + 1) * cp);
      s = D4F(2) * uld(M.f_2, q) * g3v * s23o;
      s = s + D4F(0) * uld(M.f_2, q - 2) * g3v * s23m2;
      s = s + D4F(1) * uld(M.f_2, q - 1) * g3v * s23m1;
      s = s + D4F(3) * uld(M.f_2, q + 1) * g3v * s23p1;
      s = s + D4F(1) * uld(M.f_1, q) * g3v * s13x[1];
      s = s + D4F(0) * uld(M.f_1, q - fr) * g3v * s13x[0];
      s = s + D4F(2) * uld(M.f_1, q + fr) * g3v * s13x[2];
      s = s + D4F(3) * uld(M.f_1, q + 2 * fr) * g3v * s13x[3];
      s = add_dz(s, L + (CW + 2) * cp);
      s = s - uld(M.f1_c, q) * z13;
      s = s - uld(M.f2_c, q) * z23;
      if (out) ST::st(A.u3, p, (A.a * x + Ai3 * s) * f_dcrj, A.iu3);
    }
    rm_k1 = r_k1;
    rm_k = r_k;
    rm_j = r_j;
  }
}

// ---------------------------------------------------------------------------
// Stress with coarse-grained Q: dtopo_str_111 / dtopo_str_112.
template <class ST>
struct TopoStrArgs {
  typename ST::T *xx, *yy, *zz, *xy, *xz, *yz, *r1, *r2, *r3, *r4, *r5, *r6;
  TField<ST> u1, v1, w1;
  const float *lam, *mu, *qp, *coeff, *qs, *dcrjx, *dcrjy, *dcrjz, *vx1, *vx2, *wwo;
  const int* ww;
  TMetrics M;
  WaveScales W;
  float DT, dth, dh1;
};

// The corners (j, k), (j-1, k), (j, k-1), (j-1, k-1) of one plane's 8-cell mean.
struct Corner4 {
  float c, jm, km, jk;
};
struct TopoMedium {
  Corner4 lam, mu, qp, qs;
};
__device__ __forceinline__ Corner4 corner4(const float* a, int pos, int yl) {
  return Corner4{a[pos], a[pos - yl], a[pos - 1], a[pos - yl - 1]};
}
template <class ST>
__device__ __forceinline__ TopoMedium topo_medium(const TopoStrArgs<ST>& A, int pos, int yl) {
  return TopoMedium{corner4(A.lam, pos, yl), corner4(A.mu, pos, yl), corner4(A.qp, pos, yl),
                    corner4(A.qs, pos, yl)};
}
__device__ __forceinline__ float sum8(const Corner4& a, const Corner4& b) {
  return a.c + b.c + a.jm + b.jm + a.km + b.km + a.jk + b.jk;
}

// The material averages, Q weights and the memory-variable recursion, shared
// by the one-pass kernel and the second pass (stress_attenuation.cu:200-327,
// 462-467, 534-540, 595-600, 651-656).
// m0, m1: the medium at planes i and i+1; f_vx1, f_vx2, f_wwo, ca, cb: the
// cell's relaxation texture; r_wwo = awp_rcp(f_wwo).
template <class ST>
__device__ __forceinline__ void topo_str_update(const TopoStrArgs<ST>& A, int pos, float f_dcrj,
                                                const TopoMedium& m0, const TopoMedium& m1,
                                                float nvs1, float nvs2, float nvs3, float xyv,
                                                float xzv, float yzv, float f_vx1, float f_vx2,
                                                float f_wwo, float r_wwo, float ca, float cb) {
  float xm = awp_pow2_div(16.0f, sum8(m0.mu, m1.mu));
  float xl = awp_pow2_div(8.0f, sum8(m0.lam, m1.lam)) + xm;
  float xmu1 = awp_pow2_div(2.0f, m0.mu.c + m0.mu.km);
  float xmu2 = awp_pow2_div(2.0f, m0.mu.c + m0.mu.jm);
  float xmu3 = awp_pow2_div(2.0f, m0.mu.c + m1.mu.c);
  float qpa = 0.0625f * sum8(m0.qp, m1.qp);
  const float qpaw = awp_qw_new(qpa, ca, cb, f_wwo, r_wwo, true);
  float h = 0.0625f * sum8(m0.qs, m1.qs);
  const float hw = awp_qw_new(h, ca, cb, f_wwo, r_wwo, false);
  float h1 = 0.250f * (m0.qs.c + m0.qs.km);
  const float h1w = awp_qw_new(h1, ca, cb, f_wwo, r_wwo, false);
  float h2 = 0.250f * (m0.qs.c + m0.qs.jm);
  const float h2w = awp_qw_new(h2, ca, cb, f_wwo, r_wwo, false);
  float h3 = 0.250f * (m0.qs.c + m1.qs.c);
  const float h3w = awp_qw_new(h3, ca, cb, f_wwo, r_wwo, false);
  const float DT = A.DT, dth = A.dth, dh1 = A.dh1;
  h = -xm * hw * dh1;
  h1 = -xmu1 * h1w * dh1;
  h2 = -xmu2 * h2w * dh1;
  h3 = -xmu3 * h3w * dh1;
  qpa = -qpaw * xl * dh1;
  xm = xm * dth;
  xmu1 = xmu1 * dth;
  xmu2 = xmu2 * dth;
  xmu3 = xmu3 * dth;
  xl = xl * dth;
  h = h * f_vx1;
  h1 = h1 * f_vx1;
  h2 = h2 * f_vx1;
  h3 = h3 * f_vx1;
  qpa = qpa * f_vx1;
  xm = xm + DT * h;
  xmu1 = xmu1 + DT * h1;
  xmu2 = xmu2 + DT * h2;
  xmu3 = xmu3 + DT * h3;
  const float vx1 = DT * (1 + f_vx2 * f_vx1);
  const WaveScales& W = A.W;

  const float vs1 = nvs1, vs2 = nvs2, vs3 = nvs3;
  float tmp = xl * (vs1 + vs2 + vs3);
  const float a1 = qpa * (vs1 + vs2 + vs3);
  tmp = tmp + DT * a1;
  float f_r, f_rtmp, sv;

  f_r = ST::ld(A.r1, pos, W.s[AWP_SR1]);
  f_rtmp = -h * (vs2 + vs3) + a1;
  sv = ST::ld(A.xx, pos, W.s[AWP_SXX]) + tmp - xm * (vs2 + vs3) + vx1 * f_r;
  ST::st(A.r1, pos, f_vx2 * f_r + f_wwo * f_rtmp, W.inv[AWP_SR1]);
  f_rtmp = f_rtmp * (f_wwo - 1) + f_vx2 * f_r * (1 - f_vx1);
  ST::st(A.xx, pos, (sv + DT * f_rtmp) * f_dcrj, W.inv[AWP_SXX]);

  f_r = ST::ld(A.r2, pos, W.s[AWP_SR2]);
  f_rtmp = -h * (vs1 + vs3) + a1;
  sv = (ST::ld(A.yy, pos, W.s[AWP_SYY]) + tmp - xm * (vs1 + vs3) + vx1 * f_r) * f_dcrj;
  ST::st(A.r2, pos, f_vx2 * f_r + f_wwo * f_rtmp, W.inv[AWP_SR2]);
  f_rtmp = f_rtmp * (f_wwo - 1) + f_vx2 * f_r * (1 - f_vx1);
  ST::st(A.yy, pos, (sv + DT * f_rtmp) * f_dcrj, W.inv[AWP_SYY]);

  f_r = ST::ld(A.r3, pos, W.s[AWP_SR3]);
  f_rtmp = -h * (vs1 + vs2) + a1;
  sv = (ST::ld(A.zz, pos, W.s[AWP_SZZ]) + tmp - xm * (vs1 + vs2) + vx1 * f_r) * f_dcrj;
  ST::st(A.r3, pos, f_vx2 * f_r + f_wwo * f_rtmp, W.inv[AWP_SR3]);
  f_rtmp = f_rtmp * (f_wwo - 1.0f) + f_vx2 * f_r * (1.0f - f_vx1);
  ST::st(A.zz, pos, (sv + DT * f_rtmp) * f_dcrj, W.inv[AWP_SZZ]);

  f_r = ST::ld(A.r4, pos, W.s[AWP_SR4]);
  f_rtmp = h1 * xyv;
  sv = ST::ld(A.xy, pos, W.s[AWP_SXY]) + xmu1 * xyv + vx1 * f_r;
  ST::st(A.r4, pos, f_vx2 * f_r + f_wwo * f_rtmp, W.inv[AWP_SR4]);
  f_rtmp = f_rtmp * (f_wwo - 1) + f_vx2 * f_r * (1 - f_vx1);
  ST::st(A.xy, pos, (sv + DT * f_rtmp) * f_dcrj, W.inv[AWP_SXY]);

  f_r = ST::ld(A.r5, pos, W.s[AWP_SR5]);
  f_rtmp = h2 * xzv;
  sv = ST::ld(A.xz, pos, W.s[AWP_SXZ]) + xmu2 * xzv + vx1 * f_r;
  ST::st(A.r5, pos, f_vx2 * f_r + f_wwo * f_rtmp, W.inv[AWP_SR5]);
  f_rtmp = f_rtmp * (f_wwo - 1.0f) + f_vx2 * f_r * (1.0f - f_vx1);
  ST::st(A.xz, pos, (sv + DT * f_rtmp) * f_dcrj, W.inv[AWP_SXZ]);

  f_r = ST::ld(A.r6, pos, W.s[AWP_SR6]);
  f_rtmp = h3 * yzv;
  sv = ST::ld(A.yz, pos, W.s[AWP_SYZ]) + xmu3 * yzv + vx1 * f_r;
  ST::st(A.r6, pos, f_vx2 * f_r + f_wwo * f_rtmp, W.inv[AWP_SR6]);
  f_rtmp = f_rtmp * (f_wwo - 1.0f) + f_vx2 * f_r * (1.0f - f_vx1);
  ST::st(A.yz, pos, (sv + DT * f_rtmp) * f_dcrj, W.inv[AWP_SYZ]);
}

// Stress: dtopo_str_111 (stress_attenuation.cu:74-668) on levels
// 3 <= k < nz-6 and dtopo_str_112 (:670-1410) on the top six, in one kernel
// with the velocity kernel's lane map (a chunk of nseg waves = (j, 64*nseg
// levels), march along i, ch-6 output levels per chunk, the top rows in the
// last chunk).
//
// The metric terms need 7-point (top rows: 9-point table) z sums of
// velocity columns at x neighbours (i-2 .. i+2) and y neighbours (j-2 .. j+2).
// The x-neighbour sums ride in register windows: one new column's sum per
// field and plane.  The y-neighbour sums and the own column's z differences
// read velocity columns that each plane stages in LDS (15 columns per chunk
// and row).
#define ST_NC 15
#define TOPO_NRATES AWP_TOPO_NRATES
enum {
  C_UN, C_UO, C_UM1, C_UP1, C_UP2,   // u1 at (i+2, j), (i, j), (i, j-1), (i, j+1), (i, j+2)
  C_VN, C_VO, C_VM2, C_VM1, C_VP1,   // v1 at (i+1, j), (i, j), (i, j-2), (i, j-1), (i, j+1)
  C_WN, C_WO, C_WM1, C_WP1, C_WP2    // w1 at (i+1, j), (i, j), (i, j-1), (i, j+1), (i, j+2)
};
template <class ST>
__global__ __launch_bounds__(64 * VT_MAXW) void topo_str_kernel(const TopoStrArgs<ST> A,
                                                              const TGeom G, const VelTiles V) {
  // [parity][row][column][level of the chunk]: 2 * rj * ST_NC * ch floats; the
  // column of array c at parity base L
#define LCOL(c) (L + (c) * V.ch)
  extern __shared__ float st_lds[];
  const int lane = (int)threadIdx.x;
  const int w = (int)threadIdx.y;
  const int seg = w % V.nseg, row = w / V.nseg;
  const int t = (int)blockIdx.x;
  const bool top = t == V.nint;
  const int k0 = top ? V.ktop0 : V.step * t;
  const int kl = seg * 64 + lane;  // level within the chunk: the LDS index
  const int k = k0 + kl;  // topographic level
  const int nz = G.nz;
  const int w0 = top ? V.wtop0 : V.step * t + 3;
  const int w1 = top ? nz : (V.step * t + V.ch - 3 < V.wtop0 ? V.step * t + V.ch - 3 : V.wtop0);
  const bool bnd = k >= nz - 6;
  const int kb = nz - 1 - k;  // table row of a top level
  const int jw = G.bj + (int)blockIdx.y * V.rj + row;
  const bool jok = jw < G.ej;
  const int j = __builtin_amdgcn_readfirstlane(jok ? jw : G.ej - 1);
  const int ib = G.bi + (int)blockIdx.z * V.ichunk;
  const int ie = ib + V.ichunk < G.ei ? ib + V.ichunk : G.ei;
  if (ib >= ie) return;  // uniform over the workgroup
  const bool out = k >= w0 && k < w1 && jok;
  const int sl = G.sl, yl = G.yl, fr = G.frow;
  const int kr = k < 0 ? 0 : k;          // read level (see topo_vel_kernel)
  const int K = kr + AWP_ALIGN;          // array level
  const TMetrics& M = A.M;
  const int lb = nz - 1 - k0;            // LDS level of nz-1 (top chunk)

  constexpr float phdz4[7] = {(float)TS_PHDZ4[0], (float)TS_PHDZ4[1], (float)TS_PHDZ4[2],
                              (float)TS_PHDZ4[3], (float)TS_PHDZ4[4], (float)TS_PHDZ4[5],
                              (float)TS_PHDZ4[6]};
  constexpr float pdhz4[7] = {(float)TS_PDHZ4[0], (float)TS_PDHZ4[1], (float)TS_PDHZ4[2],
                              (float)TS_PDHZ4[3], (float)TS_PDHZ4[4], (float)TS_PDHZ4[5],
                              (float)TS_PDHZ4[6]};
  // z sums of an LDS column at this lane's level
  auto zasc = [&](const float* c) {  // phdz4, ascending (normal stresses)
    float acc = phdz4[0] * c[kl - 3];
#pragma unroll
    for (int m = 1; m < 7; ++m) acc = acc + phdz4[m] * c[kl + m - 3];
    return acc;
  };
  auto zmid = [&](const float(&cf)[7], const float* c) {  // order 3, 0, 1, 2, 4, 5, 6
    float acc = cf[3] * c[kl];
    acc = acc + cf[0] * c[kl - 3];
    acc = acc + cf[1] * c[kl - 2];
    acc = acc + cf[2] * c[kl - 1];
    acc = acc + cf[4] * c[kl + 1];
    acc = acc + cf[5] * c[kl + 2];
    acc = acc + cf[6] * c[kl + 3];
    return acc;
  };
  auto zrow = [&](const FTab<6, 9>& tab, const float* c) {  // top rows, m = 8 .. 0
    float acc = tab.v[kb][8] * c[lb - 8];
#pragma unroll
    for (int m = 7; m >= 0; --m) acc = acc + tab.v[kb][m] * c[lb - m];
    return acc;
  };
  // the three x-group sums of this lane for a staged column (non-output
  // lanes compute nothing: their neighbours may lie outside the segment)
  auto zu_x = [&](const float* c) { return !out ? 0.f : (bnd ? zrow(c_str_phdz4r, c) : zasc(c)); };
  auto zv_x = [&](const float* c) { return !out ? 0.f : (bnd ? zrow(c_str_phdz4r, c) : zmid(phdz4, c)); };
  auto zw = [&](const float* c) { return !out ? 0.f : (bnd ? zrow(c_str_pdhz4r, c) : zmid(pdhz4, c)); };

  const int colj = yl * j + K;  // level K of column (i = 0, j)
  // raw x windows at this level: u (i-1 .. i+2), v and w (i-2 .. i+1), and
  // the x-group z sums Zu (i-1 .. i+2), Zv, Zw (i-2 .. i+1)
  float ux[4], vx[4], wx[4], Zu[4], Zv[4], Zw[4];
  // prologue: stage the columns the first plane's windows need
  for (int q = 0; q < 3; ++q) {
    const int iu = ib - 1 + q, iv = ib - 2 + q;
    float* L = st_lds + ((q & 1) * V.rj + row) * ST_NC * V.ch;
    ux[q + 1] = A.u1[colj + sl * iu];
    vx[q + 1] = A.v1[colj + sl * iv];
    wx[q + 1] = A.w1[colj + sl * iv];
    LCOL(C_UN)[kl] = ux[q + 1];
    LCOL(C_VN)[kl] = vx[q + 1];
    LCOL(C_WN)[kl] = wx[q + 1];
    // one-wave chunks read only their own LDS rows (see topo_vel_kernel)
    if (V.wsync && V.nseg == 1)
      wave_lds_sync();
    else
      __syncthreads();
    Zu[q + 1] = zu_x(LCOL(C_UN));
    Zv[q + 1] = zv_x(LCOL(C_VN));
    Zw[q + 1] = zw(LCOL(C_WN));
  }

  const float g_ck = M.g_c[K], g_k = M.g[K], g3c_k = M.g3_c[K], g3_k = M.g3[K];
  const float g3c_k6 = M.g3_c[bnd ? K : K + 6];  // dtopo_str_111 reads six levels up
  const float dcz = A.dcrjz[K];
  const float dcy = A.dcrjy[j];

  for (int i = ib; i < ie; ++i) {
    const int par = (i + 1) & 1;  // the prologue used parities 0, 1, 0
    float* L = st_lds + (par * V.rj + row) * ST_NC * V.ch;
    const int pos = colj + sl * i;
#pragma unroll
    for (int q = 0; q < 3; ++q) {
      ux[q] = ux[q + 1];
      vx[q] = vx[q + 1];
      wx[q] = wx[q + 1];
      Zu[q] = Zu[q + 1];
      Zv[q] = Zv[q + 1];
      Zw[q] = Zw[q + 1];
    }
    ux[3] = A.u1[pos + 2 * sl];
    vx[3] = A.v1[pos + sl];
    wx[3] = A.w1[pos + sl];
    const float um1 = A.u1[pos - yl], up1 = A.u1[pos + yl], up2 = A.u1[pos + 2 * yl];
    const float wm1 = A.w1[pos - yl], wp1 = A.w1[pos + yl], wp2 = A.w1[pos + 2 * yl];
    const float vm2 = A.v1[pos - 2 * yl], vm1 = A.v1[pos - yl], vp1 = A.v1[pos + yl];
    const float uo = ux[1], vo = vx[2], wo = wx[2];
    auto stage = [&](int c, float x) { LCOL(c)[kl] = x; };
    stage(C_UN, ux[3]);
    stage(C_UO, uo);
    stage(C_UM1, um1);
    stage(C_UP1, up1);
    stage(C_UP2, up2);
    stage(C_VN, vx[3]);
    stage(C_VO, vo);
    stage(C_VM2, vm2);
    stage(C_VM1, vm1);
    stage(C_VP1, vp1);
    stage(C_WN, wx[3]);
    stage(C_WO, wo);
    stage(C_WM1, wm1);
    stage(C_WP1, wp1);
    stage(C_WP2, wp2);
    if (V.wsync && V.nseg == 1)
      wave_lds_sync();
    else
      __syncthreads();
    Zu[3] = zu_x(LCOL(C_UN));
    Zv[3] = zv_x(LCOL(C_VN));
    Zw[3] = zw(LCOL(C_WN));
    if (out) {
      const int q = j + AWP_ALIGN + i * fr;
      const float f_dcrj = A.dcrjx[i] * dcy * dcz;
      float vs1 = 0.f, vs2 = 0.f, vs3 = 0.f, xyv = 0.f, xzv = 0.f, yzv = 0.f;
      {
        float acc;
        // xx, yy, zz
        float Jii = M.f_c[q] * g3c_k;
        Jii = awp_quot(1.0f, Jii);
        if (!bnd) {
          acc = P4F(0) * M.f1_1[q - fr] * Zu[0];
          acc = acc + P4F(1) * M.f1_1[q] * Zu[1];
        } else {
          acc = P4F(1) * M.f1_1[q] * Zu[1];
          acc = acc + P4F(0) * M.f1_1[q - fr] * Zu[0];
        }
        acc = acc + P4F(2) * M.f1_1[q + fr] * Zu[2];
        acc = acc + P4F(3) * M.f1_1[q + 2 * fr] * Zu[3];
        vs1 = D4F(1) * ux[1] + D4F(0) * ux[0] + D4F(2) * ux[2] + D4F(3) * ux[3] -
                          Jii * g_ck * acc;
        const float zv_o = bnd ? zrow(c_str_phdz4r, LCOL(C_VO)) : zasc(LCOL(C_VO));
        const float zv_m2 = bnd ? zrow(c_str_phdz4r, LCOL(C_VM2)) : zasc(LCOL(C_VM2));
        const float zv_m1 = bnd ? zrow(c_str_phdz4r, LCOL(C_VM1)) : zasc(LCOL(C_VM1));
        const float zv_p1 = bnd ? zrow(c_str_phdz4r, LCOL(C_VP1)) : zasc(LCOL(C_VP1));
        acc = P4F(2) * M.f2_2[q] * zv_o;
        acc = acc + P4F(0) * M.f2_2[q - 2] * zv_m2;
        acc = acc + P4F(1) * M.f2_2[q - 1] * zv_m1;
        acc = acc + P4F(3) * M.f2_2[q + 1] * zv_p1;
        vs2 = D4F(2) * vo + D4F(0) * vm2 + D4F(1) * vm1 + D4F(3) * vp1 -
                          Jii * g_ck * acc;
        if (!bnd) {
          const float* c = LCOL(C_WO);
          vs3 = Jii * (D4F(2) * c[kl] + D4F(0) * c[kl - 2] + D4F(1) * c[kl - 1] +
                       D4F(3) * c[kl + 1]);
        } else {
          const float* c = LCOL(C_WO);
          float zs = c_str_dhz4r.v[kb][7] * c[lb - 7];
  #pragma unroll
          for (int m = 6; m >= 0; --m) zs = zs + c_str_dhz4r.v[kb][m] * c[lb - m];
          vs3 = Jii * zs;
        }
      }
      {
        float acc;
        // xy
        float J12i = M.f[q] * g3c_k6;
        J12i = awp_quot(1.0f, J12i);
        const float zu_o = bnd ? zrow(c_str_phdz4r, LCOL(C_UO)) : zmid(phdz4, LCOL(C_UO));
        const float zu_m1 = bnd ? zrow(c_str_phdz4r, LCOL(C_UM1)) : zmid(phdz4, LCOL(C_UM1));
        const float zu_p1 = bnd ? zrow(c_str_phdz4r, LCOL(C_UP1)) : zmid(phdz4, LCOL(C_UP1));
        const float zu_p2 = bnd ? zrow(c_str_phdz4r, LCOL(C_UP2)) : zmid(phdz4, LCOL(C_UP2));
        acc = P4F(1) * M.f2_1[q] * zu_o;
        acc = acc + P4F(0) * M.f2_1[q - 1] * zu_m1;
        acc = acc + P4F(2) * M.f2_1[q + 1] * zu_p1;
        acc = acc + P4F(3) * M.f2_1[q + 2] * zu_p2;
        const float xyv1 = D4F(1) * uo + D4F(0) * um1 + D4F(2) * up1 + D4F(3) * up2 -
                           J12i * g_ck * acc;
        acc = P4F(2) * M.f1_2[q] * Zv[2];
        acc = acc + P4F(0) * M.f1_2[q - 2 * fr] * Zv[0];
        acc = acc + P4F(1) * M.f1_2[q - fr] * Zv[1];
        acc = acc + P4F(3) * M.f1_2[q + fr] * Zv[3];
        const float xyv2 = D4F(2) * vx[2] + D4F(0) * vx[0] + D4F(1) * vx[1] + D4F(3) * vx[3] -
                           J12i * g_ck * acc;
        // the update uses the shear terms only as the sums xyv1 + xyv2,
        // xzv1 + xzv2 and yzv1 + yzv2 (stress_attenuation.cu:306-327)
        xyv = xyv1 + xyv2;
      }
      {
        float acc;
        // xz
        float J13i = M.f_1[q] * g3_k;
        J13i = awp_quot(1.0f, J13i);
        float xzv1;
        if (!bnd) {
          const float* c = LCOL(C_UO);
          xzv1 = J13i * (D4F(1) * c[kl] + D4F(0) * c[kl - 1] + D4F(2) * c[kl + 1] +
                         D4F(3) * c[kl + 2]);
        } else {
          const float* c = LCOL(C_UO);
          float zs = c_str_dz4r.v[kb][6] * c[lb - 6];
  #pragma unroll
          for (int m = 5; m >= 0; --m) zs = zs + c_str_dz4r.v[kb][m] * c[lb - m];
          xzv1 = J13i * zs;
        }
        acc = P4F(2) * M.f1_c[q] * Zw[2];
        acc = acc + P4F(0) * M.f1_c[q - 2 * fr] * Zw[0];
        acc = acc + P4F(1) * M.f1_c[q - fr] * Zw[1];
        acc = acc + P4F(3) * M.f1_c[q + fr] * Zw[3];
        const float xzv2 = D4F(2) * wx[2] + D4F(0) * wx[0] + D4F(1) * wx[1] + D4F(3) * wx[3] -
                           J13i * g_k * acc;
        // yz
        float J23i = M.f_2[q] * g3_k;
        J23i = awp_quot(1.0f, J23i);
        float yzv1;
        if (!bnd) {
          const float* c = LCOL(C_VO);
          yzv1 = J23i * (D4F(1) * c[kl] + D4F(0) * c[kl - 1] + D4F(2) * c[kl + 1] +
                         D4F(3) * c[kl + 2]);
        } else {
          const float* c = LCOL(C_VO);
          float zs = c_str_dz4r.v[kb][6] * c[lb - 6];
  #pragma unroll
          for (int m = 5; m >= 0; --m) zs = zs + c_str_dz4r.v[kb][m] * c[lb - m];
          yzv1 = J23i * zs;
        }
        const float zw_m1 = zw(LCOL(C_WM1)), zw_p1 = zw(LCOL(C_WP1)), zw_p2 = zw(LCOL(C_WP2));
        acc = P4F(1) * M.f2_c[q] * Zw[2];
        acc = acc + P4F(0) * M.f2_c[q - 1] * zw_m1;
        acc = acc + P4F(2) * M.f2_c[q + 1] * zw_p1;
        acc = acc + P4F(3) * M.f2_c[q + 2] * zw_p2;
        const float yzv2 = D4F(1) * wo + D4F(0) * wm1 + D4F(2) * wp1 + D4F(3) * wp2 -
                           J23i * g_k * acc;
        xzv = xzv1 + xzv2;
        yzv = yzv1 + yzv2;
      }
      const float f_wwo = A.wwo[pos];
      const int f_ww = A.ww[pos];
      topo_str_update<ST>(A, pos, f_dcrj, topo_medium<ST>(A, pos, yl),
                          topo_medium<ST>(A, pos + sl, yl), vs1, vs2, vs3, xyv, xzv, yzv,
                          A.vx1[pos], A.vx2[pos], f_wwo, awp_rcp(f_wwo), A.coeff[f_ww * 2 - 2],
                          A.coeff[f_ww * 2 - 1]);
    }
  }
#undef LCOL
}

// The strain-rate pass of the two-pass update, in two launches by march
// direction.  Every shear rate is the sum of an x-group term (a 4-point
// combination along i of one velocity column's z sums) and a y-group term
// (along j); each normal rate has one of the two.  Marching along the group's
// own direction, a column's z sum is formed once, when the column enters the
// window, and carried through it.
//   AX = 0, march along i: vs1, vs3, the x part of xy, both parts of xz
//   AX = 1, march along j: vs2, the y part of xy (added to the stored x
//                          part), both parts of yz
// The z differences of the centre column (vs3, xz, yz) are formed from the
// same staged column and ride one or two planes behind it.  A cell takes 6
// seven-point and 3 four-point z sums, 6 velocity loads and 6 staged LDS
// columns in the two launches together; the one-direction form (marching
// along i for all six rates, in three launches) took 14, 3, 23 and 17, as the
// y-group terms need the sums of four j neighbours at every plane.
//
// Waves that hold one-sided rows take every sum with per-lane coefficients
// from LDS (c_rate_top), so their lanes do not diverge.
#define RT_ASC 0   // first term of each sum: phdz4 ascending,
#define RT_MID 9   // phdz4 from the middle,
#define RT_W 18    // pdhz4 from the middle,
#define RT_DZ 27   // dz4,
#define RT_DHZ 34  // dhz4
#define RT_N 42
// [term][class]: class 0..5 is the one-sided row of level nz-1-class in the
// order of zrow (the level furthest from the top first), class 6 the interior
// row in its own order, then zeros for the terms a one-sided row has more
// (they weigh the lane's own level, which an interior row weighs too).
struct RateTop {
  float v[RT_N][8];
};
constexpr RateTop rate_top() {
  RateTop T{};
  constexpr int dzo[4] = {1, 0, 2, 3}, dho[4] = {2, 0, 1, 3};
  for (int t = 0; t < 9; ++t)
    for (int c = 0; c < 6; ++c) {
      T.v[RT_ASC + t][c] = T.v[RT_MID + t][c] = (float)TS_PHDZ4R[c][8 - t];
      T.v[RT_W + t][c] = (float)TS_PDHZ4R[c][8 - t];
      if (t < 7) T.v[RT_DZ + t][c] = (float)TS_DZ4R[c][6 - t];
      if (t < 8) T.v[RT_DHZ + t][c] = (float)TS_DHZ4R[c][7 - t];
    }
  for (int t = 0; t < 7; ++t) {
    T.v[RT_ASC + t][6] = (float)TS_PHDZ4[t];
    T.v[RT_MID + t][6] = (float)TS_PHDZ4[rt_mid(t)];
    T.v[RT_W + t][6] = (float)TS_PDHZ4[rt_mid(t)];
  }
  for (int t = 0; t < 4; ++t) {
    T.v[RT_DZ + t][6] = (float)TOPO_D4[dzo[t]];
    T.v[RT_DHZ + t][6] = (float)TOPO_D4[dho[t]];
  }
  return T;
}
__constant__ RateTop c_rate_top = rate_top();

template <class ST, int AX>
__global__ __launch_bounds__(64 * VT_MAXW) void topo_rates_kernel(const TopoStrArgs<ST> A,
                                                                  const TGeom G,
                                                                  const VelTiles V,
                                                                  float* __restrict__ R,
                                                                  long long rstride) {
  extern __shared__ float rt_lds[];  // [parity][row][u, v, w][VT_PAD + ch + VT_PAD]
  __shared__ float s_top[RT_N * 8];
  const int lane = (int)threadIdx.x;
  const int w = (int)threadIdx.y;
  const int seg = w % V.nseg, row = w / V.nseg;
  const int t = (int)blockIdx.x;
  const bool top = t == V.nint;
  if (top) {  // uniform over the workgroup
    for (int e = w * 64 + lane; e < RT_N * 8; e += V.nseg * V.rj * 64)
      s_top[e] = (&c_rate_top.v[0][0])[e];
    __syncthreads();
  }
  const int k0 = top ? V.ktop0 : V.step * t;
  const int kl = seg * 64 + lane;  // level within the chunk
  const int k = k0 + kl;
  const int nz = G.nz;
  const int w0 = top ? V.wtop0 : V.step * t + 3;
  const int w1 = top ? nz : (V.step * t + V.ch - 3 < V.wtop0 ? V.step * t + V.ch - 3 : V.wtop0);
  const bool bnd = k >= nz - 6;
  // whether this wave holds one-sided rows
  const bool topw = top && __builtin_amdgcn_readfirstlane(k0 + seg * 64 + 63) >= nz - 6;
  // fixed line f (j or i), march m (i or j)
  const int f0 = AX == 0 ? G.bj : G.bi, f1 = AX == 0 ? G.ej : G.ei;
  const int m1 = AX == 0 ? G.ei : G.ej;
  const int fw = f0 + (int)blockIdx.y * V.rj + row;
  const bool fok = fw < f1;
  const int f = __builtin_amdgcn_readfirstlane(fok ? fw : f1 - 1);
  const int mb = (AX == 0 ? G.bi : G.bj) + (int)blockIdx.z * V.ichunk;
  const int me = mb + V.ichunk < m1 ? mb + V.ichunk : m1;
  if (mb >= me) return;  // uniform over the workgroup
  const bool out = k >= w0 && k < w1 && fok;
  const int sm = AX == 0 ? G.sl : G.yl;     // field stride along the march
  const int fm = AX == 0 ? G.frow : 1;      // metric stride along the march
  const int K = (k < 0 ? 0 : k) + AWP_ALIGN;  // array level (see topo_vel_kernel)
  const int base = K + (AX == 0 ? G.yl : G.sl) * f;
  const int qbase = AWP_ALIGN + (AX == 0 ? 1 : G.frow) * f;
  const TMetrics& M = A.M;
  const int cp = V.ch + 2 * VT_PAD;
  const int own = VT_PAD + kl;  // this lane's level in a staged column
  const int lb = VT_PAD + nz - 1 - k0;  // level nz-1 (top chunk)
  const int cls = bnd ? nz - 1 - k : 6;

  constexpr float phdz4[7] = {(float)TS_PHDZ4[0], (float)TS_PHDZ4[1], (float)TS_PHDZ4[2],
                              (float)TS_PHDZ4[3], (float)TS_PHDZ4[4], (float)TS_PHDZ4[5],
                              (float)TS_PHDZ4[6]};
  constexpr float pdhz4[7] = {(float)TS_PDHZ4[0], (float)TS_PDHZ4[1], (float)TS_PDHZ4[2],
                              (float)TS_PDHZ4[3], (float)TS_PDHZ4[4], (float)TS_PDHZ4[5],
                              (float)TS_PDHZ4[6]};
  auto asc = [&](const float* c) {
    float acc = phdz4[0] * c[own - 3];
#pragma unroll
    for (int m = 1; m < 7; ++m) acc = acc + phdz4[m] * c[own + m - 3];
    return acc;
  };
  auto mid = [&](const float(&cf)[7], const float* c) {
    float acc = cf[3] * c[own];
#pragma unroll
    for (int m = 1; m < 7; ++m) acc = acc + cf[rt_mid(m)] * c[own + rt_mid(m) - 3];
    return acc;
  };
  // the n-term sum of table rows r0 .. r0+n-1; off(t): the interior term's level
  auto tops = [&](int r0, int n, auto off, const float* c) {
    float acc = 0.f;
#pragma unroll
    for (int m = 0; m < n; ++m) {
      const float x = s_top[(r0 + m) * 8 + cls] * c[bnd ? lb - (n - 1) + m : own + off(m)];
      acc = m == 0 ? x : acc + x;
    }
    return acc;
  };
  auto off_asc = [](int m) { return m < 7 ? m - 3 : 0; };
  auto off_mid = [](int m) { return m < 7 ? rt_mid(m) - 3 : 0; };
  auto off_dz = [](int m) { return m == 1 ? -1 : m == 2 ? 1 : m == 3 ? 2 : 0; };
  auto off_dhz = [](int m) { return m == 1 ? -2 : m == 2 ? -1 : m == 3 ? 1 : 0; };
  struct Sums {
    float zu, zv, zw, d, dw;  // d: dz of u (AX = 0) or v (AX = 1); dw: dhz of w (AX = 0)
  };
  int par = 0;
  // stage the three columns entering the windows and form their z sums
  auto enter = [&](float u, float v, float x) {
    float* cu = rt_lds + (par * V.rj + row) * 3 * cp;
    float *cv = cu + cp, *cw = cv + cp;
    par ^= 1;
    cu[own] = u;
    cv[own] = v;
    cw[own] = x;
    // one-wave chunks read only their own LDS (see topo_vel_kernel)
    if (V.wsync && V.nseg == 1)
      wave_lds_sync();
    else
      __syncthreads();
    Sums s;
    const float* cd = AX == 0 ? cu : cv;
    s.dw = 0.f;
    if (!topw) {
      s.zu = AX == 0 ? asc(cu) : mid(phdz4, cu);
      s.zv = AX == 0 ? mid(phdz4, cv) : asc(cv);
      s.zw = mid(pdhz4, cw);
      s.d = D4F(1) * cd[own] + D4F(0) * cd[own - 1] + D4F(2) * cd[own + 1] + D4F(3) * cd[own + 2];
      if (AX == 0)
        s.dw = D4F(2) * cw[own] + D4F(0) * cw[own - 2] + D4F(1) * cw[own - 1] +
               D4F(3) * cw[own + 1];
    } else {
      s.zu = AX == 0 ? tops(RT_ASC, 9, off_asc, cu) : tops(RT_MID, 9, off_mid, cu);
      s.zv = AX == 0 ? tops(RT_MID, 9, off_mid, cv) : tops(RT_ASC, 9, off_asc, cv);
      s.zw = tops(RT_W, 9, off_mid, cw);
      s.d = tops(RT_DZ, 7, off_dz, cd);
      if (AX == 0) s.dw = tops(RT_DHZ, 8, off_dhz, cw);
    }
    return s;
  };

  // windows: u covers m-1 .. m+2, v m-2 .. m+1, w m-2 .. m+1 (AX = 0) or
  // m-1 .. m+2 (AX = 1)
  constexpr int UL = -1, VL = -2, WL = AX == 0 ? -2 : -1;
  float U[4], Vv[4], W[4], ZU[4], ZV[4], ZW[4], D[3], dwc = 0.f;
  auto at = [&](int m) { return base + sm * m; };
#pragma unroll
  for (int q = 0; q < 3; ++q) {
    U[q + 1] = A.u1[at(mb + UL + q)];
    Vv[q + 1] = A.v1[at(mb + VL + q)];
    W[q + 1] = A.w1[at(mb + WL + q)];
  }
  float un = A.u1[at(mb + UL + 3)], vn = A.v1[at(mb + VL + 3)], wn = A.w1[at(mb + WL + 3)];
#pragma unroll
  for (int q = 0; q < 3; ++q) {
    const Sums s = enter(U[q + 1], Vv[q + 1], W[q + 1]);
    ZU[q + 1] = s.zu;
    ZV[q + 1] = s.zv;
    ZW[q + 1] = s.zw;
    D[q] = s.d;
    dwc = s.dw;
  }
  const float g_ck = M.g_c[K], g_k = M.g[K], g3c_k = M.g3_c[K], g3_k = M.g3[K];
  const float g3c_k6 = M.g3_c[bnd ? K : K + 6];  // dtopo_str_111 reads six levels up

  for (int m = mb; m < me; ++m) {
    const int pos = at(m);
    const int q = qbase + fm * m;
#pragma unroll
    for (int x = 0; x < 3; ++x) {
      U[x] = U[x + 1];
      Vv[x] = Vv[x + 1];
      W[x] = W[x + 1];
      ZU[x] = ZU[x + 1];
      ZV[x] = ZV[x + 1];
      ZW[x] = ZW[x + 1];
    }
    U[3] = un;
    Vv[3] = vn;
    W[3] = wn;
    // the next plane's columns; one plane past the bounds stays in the
    // padded array
    un = A.u1[at(m + 1 + UL + 3)];
    vn = A.v1[at(m + 1 + VL + 3)];
    wn = A.w1[at(m + 1 + WL + 3)];
    float xpart = 0.f;
    if (AX == 1 && out) xpart = R[3 * rstride + pos];
    const Sums s = enter(U[3], Vv[3], W[3]);
    ZU[3] = s.zu;
    ZV[3] = s.zv;
    ZW[3] = s.zw;
    // D[0..2] end at the newest column before this one: u's centre is two
    // planes behind it, v's one; w's centre is one behind
    const float dc = AX == 0 ? D[1] : D[2];
    D[0] = D[1];
    D[1] = D[2];
    D[2] = s.d;
    const float Jii = awp_pow2_div(1.0f, uld(M.f_c, q) * g3c_k);
    const float J12i = awp_pow2_div(1.0f, uld(M.f, q) * g3c_k6);
    float acc;
    if (AX == 0) {
      acc = P4F(0) * uld(M.f1_1, q - fm) * ZU[0];
      acc = acc + P4F(1) * uld(M.f1_1, q) * ZU[1];
      acc = acc + P4F(2) * uld(M.f1_1, q + fm) * ZU[2];
      acc = acc + P4F(3) * uld(M.f1_1, q + 2 * fm) * ZU[3];
      const float vs1 =
          D4F(1) * U[1] + D4F(0) * U[0] + D4F(2) * U[2] + D4F(3) * U[3] - Jii * g_ck * acc;
      const float vs3 = Jii * dwc;
      dwc = s.dw;
      acc = P4F(2) * uld(M.f1_2, q) * ZV[2];
      acc = acc + P4F(0) * uld(M.f1_2, q - 2 * fm) * ZV[0];
      acc = acc + P4F(1) * uld(M.f1_2, q - fm) * ZV[1];
      acc = acc + P4F(3) * uld(M.f1_2, q + fm) * ZV[3];
      const float xyv2 =
          D4F(2) * Vv[2] + D4F(0) * Vv[0] + D4F(1) * Vv[1] + D4F(3) * Vv[3] - J12i * g_ck * acc;
      const float J13i = awp_pow2_div(1.0f, uld(M.f_1, q) * g3_k);
      const float xzv1 = J13i * dc;
      acc = P4F(2) * uld(M.f1_c, q) * ZW[2];
      acc = acc + P4F(0) * uld(M.f1_c, q - 2 * fm) * ZW[0];
      acc = acc + P4F(1) * uld(M.f1_c, q - fm) * ZW[1];
      acc = acc + P4F(3) * uld(M.f1_c, q + fm) * ZW[3];
      const float xzv2 =
          D4F(2) * W[2] + D4F(0) * W[0] + D4F(1) * W[1] + D4F(3) * W[3] - J13i * g_k * acc;
      if (out) {
        R[pos] = vs1;
        R[2 * rstride + pos] = vs3;
        R[3 * rstride + pos] = xyv2;
        R[4 * rstride + pos] = xzv1 + xzv2;
      }
    } else {
      acc = P4F(2) * uld(M.f2_2, q) * ZV[2];
      acc = acc + P4F(0) * uld(M.f2_2, q - 2) * ZV[0];
      acc = acc + P4F(1) * uld(M.f2_2, q - 1) * ZV[1];
      acc = acc + P4F(3) * uld(M.f2_2, q + 1) * ZV[3];
      const float vs2 =
          D4F(2) * Vv[2] + D4F(0) * Vv[0] + D4F(1) * Vv[1] + D4F(3) * Vv[3] - Jii * g_ck * acc;
      acc = P4F(1) * uld(M.f2_1, q) * ZU[1];
      acc = acc + P4F(0) * uld(M.f2_1, q - 1) * ZU[0];
      acc = acc + P4F(2) * uld(M.f2_1, q + 1) * ZU[2];
      acc = acc + P4F(3) * uld(M.f2_1, q + 2) * ZU[3];
      const float xyv1 =
          D4F(1) * U[1] + D4F(0) * U[0] + D4F(2) * U[2] + D4F(3) * U[3] - J12i * g_ck * acc;
      const float J23i = awp_pow2_div(1.0f, uld(M.f_2, q) * g3_k);
      const float yzv1 = J23i * dc;
      acc = P4F(1) * uld(M.f2_c, q) * ZW[1];
      acc = acc + P4F(0) * uld(M.f2_c, q - 1) * ZW[0];
      acc = acc + P4F(2) * uld(M.f2_c, q + 1) * ZW[2];
      acc = acc + P4F(3) * uld(M.f2_c, q + 2) * ZW[3];
      const float yzv2 =
          D4F(1) * W[1] + D4F(0) * W[0] + D4F(2) * W[2] + D4F(3) * W[3] - J23i * g_k * acc;
      if (out) {
        R[rstride + pos] = vs2;
        R[3 * rstride + pos] = xyv1 + xpart;
        R[5 * rstride + pos] = yzv1 + yzv2;
      }
    }
  }
}

// The relaxation texture of the Q pass: the per-cell arrays (TOPO_TEX_ARRAYS),
// or vx1, vx2, wwo from the 8-entry table indexed by ww, with ww read
// (TOPO_TEX_TABLE) or evaluated from init_texture's parity rule
// (TOPO_TEX_RULE, mesh.c:1103-1137) over the stress region that starts at
// (xls, yls, align) and has nj columns per x plane and nzt levels.
enum { TOPO_TEX_ARRAYS = 0, TOPO_TEX_TABLE = 1, TOPO_TEX_RULE = 2 };
struct TopoTex {
  float t[24];  // vx1[8], vx2[8], wwo[8]
  int xls, yls, nj, nzt;
};

// The material averages, Q weights and memory-variable recursion of the
// stress update (topo_str_update) over the cells topo_rates_kernel wrote rates
// for: levels 3 <= k < nz of the stress bounds.  It streams 136 B per cell
// (6 rates and 4 medium arrays read, 6 stresses and 6 memory variables read
// and written), so it runs as the Cartesian stress kernel does: tiles of
// awp_pick_tile in XCD-aware order, an i-march that carries the medium's
// plane i+1 in registers.  One plane per workgroup, in the launch's own order,
// fetched the medium's neighbour planes and rows again in every XCD (1.75 GB
// per 256x256x192 update for 1.11 algorithmic).
struct TopoQLaunch {
  AwpTile tile;
  int nkt, njt, ichunk, nblocks;
};

template <class ST, int TEX>
__global__ __launch_bounds__(512) void topo_str_q_kernel(const TopoStrArgs<ST> A, const TGeom G,
                                                         const float* __restrict__ R,
                                                         long long rstride, const TopoQLaunch L,
                                                         const TopoTex TT) {
  __shared__ float s_tex[32];  // vx1[8], vx2[8], wwo[8], 1/wwo[8]
  __shared__ float s_coeff[16];
  const int tid = (int)threadIdx.x;
  if (tid < 16) s_coeff[tid] = A.coeff[tid];
  if (TEX != TOPO_TEX_ARRAYS && tid < 32)
    s_tex[tid] = tid < 24 ? TT.t[tid] : awp_rcp(TT.t[tid - 8]);
  __syncthreads();
  const int b = awp_xcd_remap((int)blockIdx.x, L.nblocks);
  int kt, jt, ic;
  awp_tile3(b, L.nkt, L.njt, 0, kt, jt, ic);
  const int lr = tid * L.tile.mul >> 20;  // row of this lane in the tile (awp_pick_tile)
  const int K = AWP_ALIGN + kt * L.tile.width + (tid - lr * L.tile.width);  // array level
  const int k = K - AWP_ALIGN;
  const int j = G.bj + jt * L.tile.rows + lr;
  if (lr >= L.tile.rows || k < 3 || k >= G.nz || j >= G.ej) return;
  const int ib = G.bi + ic * L.ichunk;
  const int ie = ib + L.ichunk < G.ei ? ib + L.ichunk : G.ei;
  const int sl = G.sl, yl = G.yl;
  const float dcz = A.dcrjz[K];
  const float dcy = A.dcrjy[j];
  int pos = yl * j + K + sl * ib;
  TopoMedium m0 = topo_medium<ST>(A, pos, yl);
  for (int i = ib; i < ie; ++i, pos += sl) {
    const TopoMedium m1 = topo_medium<ST>(A, pos + sl, yl);
    const float f_dcrj = A.dcrjx[i] * dcy * dcz;
    float f_vx1, f_vx2, f_wwo, r_wwo;
    int f_ww;
    if (TEX == TOPO_TEX_ARRAYS) {
      f_vx1 = A.vx1[pos]; f_vx2 = A.vx2[pos]; f_wwo = A.wwo[pos];
      f_ww = A.ww[pos];
      r_wwo = awp_rcp(f_wwo);
    } else {
      if (TEX == TOPO_TEX_TABLE) {
        f_ww = A.ww[pos];
      } else {
        const int ni = i - TT.xls, col = ni * TT.nj + (j - TT.yls);
        f_ww = 1 + 4 * ((ni + 1) & 1) + 2 * ((col + 1) & 1) + ((TT.nzt + col * TT.nzt + k) & 1);
      }
      const int t = (f_ww - 1) & 7;
      f_vx1 = s_tex[t]; f_vx2 = s_tex[8 + t]; f_wwo = s_tex[16 + t];
      r_wwo = s_tex[24 + t];
    }
    topo_str_update<ST>(A, pos, f_dcrj, m0, m1, R[pos], R[rstride + pos], R[2 * rstride + pos],
                        R[3 * rstride + pos], R[4 * rstride + pos], R[5 * rstride + pos],
                        f_vx1, f_vx2, f_wwo, r_wwo, s_coeff[(f_ww * 2 - 2) & 15],
                        s_coeff[(f_ww * 2 - 1) & 15]);
    m0 = m1;
  }
}

// ---------------------------------------------------------------------------
// Metrics (setup).  f* over topographic (a, b) in [-6, n+6)^2; f on [-8, n+8).
struct FPtrs {
  float *f, *f_1, *f_2, *f_c, *f1_1, *f1_2, *f1_c, *f2_1, *f2_2, *f2_c;
};

__global__ void geom_custom_kernel(float* f, int nx, int ny, int frow, float normalize) {
  const int b = -AWP_NGSL + (int)(blockIdx.x * 64 + threadIdx.x);
  const int a = -AWP_NGSL + (int)blockIdx.y;
  if (b >= ny + AWP_NGSL || a >= nx + AWP_NGSL) return;
  const int idx = (b + AWP_ALIGN + AWP_NGSL + 2) + (a + AWP_NGSL + 2) * frow;
  f[idx] = (float)(1.0 + (double)(f[idx] * normalize));
}

__global__ void metrics_interp_kernel(FPtrs F, int nx, int ny, int frow) {
  const int b = -6 + (int)(blockIdx.x * 64 + threadIdx.x);
  const int a = -6 + (int)blockIdx.y;
  if (b >= ny + 6 || a >= nx + 6) return;
  const int q = (b + AWP_ALIGN + AWP_NGSL + 2) + (a + AWP_NGSL + 2) * frow;
  const float* f = F.f;
  F.f_1[q] = P4F(0) * f[q - 2] + P4F(1) * f[q - 1] + P4F(2) * f[q] + P4F(3) * f[q + 1];
  F.f_2[q] = P4F(0) * f[q - frow] + P4F(1) * f[q] + P4F(2) * f[q + frow] + P4F(3) * f[q + 2 * frow];
  float acc = 0.f;
#pragma unroll
  for (int t = 0; t < 4; ++t) {
    const int r = q - 2 + t;
    const float row = P4F(0) * f[r - frow] + P4F(1) * f[r] + P4F(2) * f[r + frow] +
                      P4F(3) * f[r + 2 * frow];
    acc = t == 0 ? P4F(0) * row : acc + P4F(t) * row;
  }
  F.f_c[q] = acc;
}

__global__ void metrics_diff_kernel(FPtrs F, int nx, int ny, int frow, float hi) {
  const int b = -6 + (int)(blockIdx.x * 64 + threadIdx.x);
  const int a = -6 + (int)blockIdx.y;
  if (b >= ny + 6 || a >= nx + 6) return;
  const int q = (b + AWP_ALIGN + AWP_NGSL + 2) + (a + AWP_NGSL + 2) * frow;
  const int r = frow;
  const float *f = F.f, *f_1 = F.f_1, *f_2 = F.f_2, *f_c = F.f_c;
  F.f1_1[q] = hi * (D4F(0) * f_c[q - 2 * r] + D4F(1) * f_c[q - r] + D4F(2) * f_c[q] +
                    D4F(3) * f_c[q + r]);
  F.f1_2[q] = hi * (D4F(0) * f[q - r] + D4F(1) * f[q] + D4F(2) * f[q + r] + D4F(3) * f[q + 2 * r]);
  F.f1_c[q] = hi * (D4F(0) * f_1[q - r] + D4F(1) * f_1[q] + D4F(2) * f_1[q + r] +
                    D4F(3) * f_1[q + 2 * r]);
  F.f2_1[q] = hi * (D4F(0) * f[q - 2] + D4F(1) * f[q - 1] + D4F(2) * f[q] + D4F(3) * f[q + 1]);
  F.f2_2[q] = hi * (D4F(0) * f_c[q - 1] + D4F(1) * f_c[q] + D4F(2) * f_c[q + 1] +
                    D4F(3) * f_c[q + 2]);
  F.f2_c[q] = hi * (D4F(0) * f_2[q - 2] + D4F(1) * f_2[q - 1] + D4F(2) * f_2[q] +
                    D4F(3) * f_2[q + 1]);
}

// g without stretching (geom_no_grid_stretching): g(k) = h' k, 0 at the top
// ghost.
__global__ void g_fill_kernel(float* g0, int nz, float hp) {
  const int k = (int)(blockIdx.x * 64 + threadIdx.x);
  if (k >= nz) return;
  g0[AWP_ALIGN + k] = k == nz - 1 ? 0.0f : (float)((double)hp * ((double)k - 0.5 * 0 - 0));
}

// g_c, then g3 and g3_c; one workgroup, two passes.
__global__ __launch_bounds__(256) void metrics_g_kernel(const float* g0, float* gc0, float* g30,
                                                        float* g3c0, int nz, float hi) {
  const float* G = g0 + AWP_ALIGN;
  float* Gc = gc0 + AWP_ALIGN;
  float* G3 = g30 + AWP_ALIGN;
  float* G3c = g3c0 + AWP_ALIGN;
  for (int k = (int)threadIdx.x; k < nz; k += 256) {
    float acc;
    if (k < 6) {
      acc = (float)TM_PHZL[k][0] * G[0];
      for (int m = 1; m < 7; ++m) acc = acc + (float)TM_PHZL[k][m] * G[m];
    } else if (k >= nz - 6) {
      const int r = nz - 1 - k;
      acc = (float)TM_PHZR[r][7] * G[nz - 8];
      for (int m = 6; m >= 0; --m) acc = acc + (float)TM_PHZR[r][m] * G[nz - 1 - m];
    } else {
      acc = P4F(0) * G[k - 2] + P4F(1) * G[k - 1] + P4F(2) * G[k] + P4F(3) * G[k + 1];
    }
    Gc[k] = acc;
  }
  __syncthreads();
  for (int k = (int)threadIdx.x; k < nz; k += 256) {
    float acc, accc;
    if (k < 6) {
      acc = (float)TM_DZL[k][0] * Gc[0];
      for (int m = 1; m < 8; ++m) acc = acc + (float)TM_DZL[k][m] * Gc[m];
      accc = (float)TM_DHZL[k][0] * G[0];
      for (int m = 1; m < 7; ++m) accc = accc + (float)TM_DHZL[k][m] * G[m];
    } else if (k >= nz - 6) {
      const int r = nz - 1 - k;
      acc = (float)TM_DZR[r][6] * Gc[nz - 7];
      for (int m = 5; m >= 0; --m) acc = acc + (float)TM_DZR[r][m] * Gc[nz - 1 - m];
      accc = (float)TM_DHZR[r][7] * G[nz - 8];
      for (int m = 6; m >= 0; --m) accc = accc + (float)TM_DHZR[r][m] * G[nz - 1 - m];
    } else {
      acc = D4F(0) * Gc[k - 1] + D4F(1) * Gc[k] + D4F(2) * Gc[k + 1] + D4F(3) * Gc[k + 2];
      accc = D4F(0) * G[k - 2] + D4F(1) * G[k - 1] + D4F(2) * G[k] + D4F(3) * G[k + 1];
    }
    G3[k] = k == nz - 1 ? 1.0f : hi * acc;
    G3c[k] = hi * accc;
  }
}

// ---------------------------------------------------------------------------
// Host side.
// The stress kernels' constants (set_constants, stress_attenuation.cu:39-72),
// process-wide like the reference's __constant__ block.
struct TopoConstants {
  float DT, dth, dh1;
  int set;
};
TopoConstants g_topo_constants = {0.0f, 0.0f, 0.0f, 0};

bool topo_geom(const topo_t* T, const char* where, TGeom* G) {
  if (!T) {
    awp_set_error(AWP_ERR_ARG, "%s: topo_t is NULL", where);
    return false;
  }
  if (T->nx < 8 || T->ny < 8 || T->nz < 18) {
    awp_set_error(AWP_ERR_ARG, "%s: grid %d x %d x %d too small (need nx, ny >= 8, nz >= 18)",
                  where, T->nx, T->ny, T->nz);
    return false;
  }
  const long long yl = T->nz + 2 * AWP_ALIGN;
  const long long sl = (long long)(T->ny + 4 + AWP_NGSL2) * yl;
  const long long n = sl * (T->nx + 4 + AWP_NGSL2);
  if (n * 2 >= (1ll << 31)) {
    awp_set_error(AWP_ERR_ARG, "%s: %lld cells per field exceed the 32-bit index range", where,
                  n);
    return false;
  }
  G->nx = T->nx;
  G->ny = T->ny;
  G->nz = T->nz;
  G->yl = (int)yl;
  G->sl = (int)sl;
  G->frow = 2 * AWP_ALIGN + 2 * AWP_NGSL + T->ny + 4;
  return true;
}

TMetrics topo_metrics(const topo_t* T) {
  const f_grid_t& f = T->metrics_f;
  const g_grid_t& g = T->metrics_g;
  TMetrics M;
  M.f = f.d_f;
  M.f_1 = f.d_f_1;
  M.f_2 = f.d_f_2;
  M.f_c = f.d_f_c;
  M.f1_1 = f.d_f1_1;
  M.f1_2 = f.d_f1_2;
  M.f1_c = f.d_f1_c;
  M.f2_1 = f.d_f2_1;
  M.f2_2 = f.d_f2_2;
  M.f2_c = f.d_f2_c;
  M.g = g.d_g;
  M.g3 = g.d_g3;
  M.g3_c = g.d_g3_c;
  M.g_c = g.d_g_c;
  return M;
}

bool metrics_present(const TMetrics& M, const char* where) {
  const float* all[14] = {M.f, M.f_1, M.f_2, M.f_c, M.f1_1, M.f1_2, M.f1_c,
                          M.f2_1, M.f2_2, M.f2_c, M.g, M.g3, M.g3_c, M.g_c};
  for (const float* x : all)
    if (!x) {
      awp_set_error(AWP_ERR_ARG, "%s: a metric array is NULL", where);
      return false;
    }
  return true;
}

// Chunks of the curvilinear kernels' k lane map for a column of nz levels:
// nseg = ceil(nz / 64) waves of 64 levels per chunk, at most `most` and
// topo_nseg, so a column of up to 64 * nseg levels is one chunk (nz = 192: three
// waves, where one-wave segments of 58 outputs need four, one of them with 12).
// The velocity kernel takes chunks of 2 to 4 waves (one-wave segments at
// 160x160x128 81 against 60 us, at 160x160x256 132 / 118) and one-wave segments
// on columns of more than 256 levels: all waves of a chunk meet at every plane,
// and with 5 to 8 of them 160x160x257 took 228 against 140 us, 256x256x320 610 /
// 391 and 256x256x520 958 / 560.
void topo_tiles(int nz, int most, VelTiles* V) {
  int nseg = awp_cdiv(nz, 64);
  const int cap = awp_tuning().topo_nseg;
  if (nseg > most) nseg = most;
  if (nseg > cap) nseg = cap;
  if (nseg > VT_MAXW) nseg = VT_MAXW;
  if (nseg < 1) nseg = 1;
  V->nseg = nseg;
  V->ch = 64 * nseg;
  V->step = V->ch - 6;
  // one j row per workgroup for chunks, so each plane's barrier waits only
  // for the chunk's own waves (1.87 -> 1.78 ms per stress update at
  // 384x384x192 against two rows); four rows of one-wave segments
  V->rj = nseg == 1 ? 4 : 1;
  const int rjf = awp_tuning().topo_rj;  // > 0 forces the rows per workgroup
  if (rjf > 0) V->rj = rjf * nseg <= VT_MAXW ? rjf : VT_MAXW / nseg;
  if (V->rj < 1) V->rj = 1;
  V->ktop0 = nz - V->ch;
  V->wtop0 = V->ktop0 + 3 > 3 ? V->ktop0 + 3 : 3;
  V->nint = V->wtop0 > 3 ? awp_cdiv(V->wtop0 - 3, V->step) : 0;
}

// Planes per march of a velocity or strain-rate launch whose planes take
// `waves` waves each: 4 to `most`, the count that minimises rounds x (planes +
// 3).  The card holds 4096 of these waves at a time (4 per SIMD: 108 to 127
// VGPRs), a last round that is nearly empty takes as long as a full one, and a
// march first loads and sums 3 planes for its windows.  At 131x97x85 the
// velocity update takes 41 us with 6 planes (4268 waves), 31 with 8 (3298).
int topo_chunk(int planes, int waves, int most, int forced) {
  if (forced > 0) return forced;
  int best = 4;
  long long cost = 1ll << 62;
  for (int c = 4; c <= most; ++c) {
    const long long w = (long long)awp_cdiv(planes, c) * waves;
    const long long x = (w + 4095) / 4096 * (c + 3);
    if (x < cost) {
      cost = x;
      best = c;
    }
  }
  return best;
}

template <class ST>
void topo_velocity_launch(topo_t* T, const WaveScales& W, const char* where) {
  TGeom G;
  if (!topo_geom(T, where, &G)) return;
  if (!T->use) return;
  TopoVelArgs<ST> A;
  using Q = typename ST::T;
  A.u1 = reinterpret_cast<Q*>(T->u1);
  A.u2 = reinterpret_cast<Q*>(T->v1);
  A.u3 = reinterpret_cast<Q*>(T->w1);
  A.s11 = TField<ST>{reinterpret_cast<const Q*>(T->xx), W.s[AWP_SXX]};
  A.s12 = TField<ST>{reinterpret_cast<const Q*>(T->xy), W.s[AWP_SXY]};
  A.s13 = TField<ST>{reinterpret_cast<const Q*>(T->xz), W.s[AWP_SXZ]};
  A.s22 = TField<ST>{reinterpret_cast<const Q*>(T->yy), W.s[AWP_SYY]};
  A.s23 = TField<ST>{reinterpret_cast<const Q*>(T->yz), W.s[AWP_SYZ]};
  A.s33 = TField<ST>{reinterpret_cast<const Q*>(T->zz), W.s[AWP_SZZ]};
  A.su1 = W.s[AWP_SU];
  A.su2 = W.s[AWP_SV];
  A.su3 = W.s[AWP_SW];
  A.iu1 = W.inv[AWP_SU];
  A.iu2 = W.inv[AWP_SV];
  A.iu3 = W.inv[AWP_SW];
  A.rho = T->rho;
  A.dcrjx = T->dcrjx;
  A.dcrjy = T->dcrjy;
  A.dcrjz = T->dcrjz;
  A.M = topo_metrics(T);
  A.a = T->timestep;
  A.nu = T->dth;
  if (!metrics_present(A.M, where)) return;
  if (!T->u1 || !T->v1 || !T->w1 || !T->xx || !T->yy || !T->zz || !T->xy || !T->xz ||
      !T->yz || !T->rho || !T->dcrjx || !T->dcrjy || !T->dcrjz) {
    awp_set_error(AWP_ERR_ARG, "%s: a field pointer is NULL", where);
    return;
  }
  // velocity bounds of one rank without neighbours: i in [0, nx), j in [0, ny)
  // (topography.c:309-335); the reference splits j into front / interior /
  // back launches of the same kernels.
  G.bi = 0;
  G.ei = T->nx;
  G.bj = 0;
  G.ej = T->ny;
  hipStream_t st = T->stream_i;
  VelTiles V;
  topo_tiles(T->nz, T->nz > 256 ? 1 : 4, &V);
  V.wsync = awp_tuning().topo_wsync;
  V.njt = awp_cdiv(T->ny, V.rj);
  V.ichunk = topo_chunk(T->nx, (V.nint + 1) * T->ny * V.nseg, 8, awp_tuning().topo_vel_ichunk);
  const dim3 block(64, V.nseg * V.rj, 1);
  const dim3 grid((V.nint + 1) * V.njt * awp_cdiv(T->nx, V.ichunk));
  const size_t lds = (size_t)2 * V.rj * VT_NL * (V.ch + 2 * VT_PAD) * sizeof(float);
  hipLaunchKernelGGL((topo_vel_kernel<ST>), grid, block, lds, st, A, G, V);
  awp_check_launch(where);
}

// tex, texmode: the Q pass's relaxation texture (TOPO_TEX_*; tex holds
// vx1[8], vx2[8], wwo[8] unless texmode is TOPO_TEX_ARRAYS, which the
// one-pass update always uses).
template <class ST>
void topo_stress_launch(topo_t* T, const WaveScales& W, const char* where, float* rates,
                        const float* tex = nullptr, int texmode = TOPO_TEX_ARRAYS) {
  TGeom G;
  if (!topo_geom(T, where, &G)) return;
  if (!T->use) return;
  if (!g_topo_constants.set) {
    awp_set_error(AWP_ERR_STATE, "%s: topo_set_constants has not been called", where);
    return;
  }
  TopoStrArgs<ST> A;
  using Q = typename ST::T;
  A.xx = reinterpret_cast<Q*>(T->xx);
  A.yy = reinterpret_cast<Q*>(T->yy);
  A.zz = reinterpret_cast<Q*>(T->zz);
  A.xy = reinterpret_cast<Q*>(T->xy);
  A.xz = reinterpret_cast<Q*>(T->xz);
  A.yz = reinterpret_cast<Q*>(T->yz);
  A.r1 = reinterpret_cast<Q*>(T->r1);
  A.r2 = reinterpret_cast<Q*>(T->r2);
  A.r3 = reinterpret_cast<Q*>(T->r3);
  A.r4 = reinterpret_cast<Q*>(T->r4);
  A.r5 = reinterpret_cast<Q*>(T->r5);
  A.r6 = reinterpret_cast<Q*>(T->r6);
  A.u1 = TField<ST>{reinterpret_cast<const Q*>(T->u1), W.s[AWP_SU]};
  A.v1 = TField<ST>{reinterpret_cast<const Q*>(T->v1), W.s[AWP_SV]};
  A.w1 = TField<ST>{reinterpret_cast<const Q*>(T->w1), W.s[AWP_SW]};
  A.lam = T->lami;
  A.mu = T->mui;
  A.qp = T->qpi;
  A.coeff = T->coeff;
  A.qs = T->qsi;
  A.dcrjx = T->dcrjx;
  A.dcrjy = T->dcrjy;
  A.dcrjz = T->dcrjz;
  A.vx1 = T->vx1;
  A.vx2 = T->vx2;
  A.ww = T->ww;
  A.wwo = T->wwo;
  A.M = topo_metrics(T);
  A.W = W;
  A.DT = g_topo_constants.DT;
  A.dth = g_topo_constants.dth;
  A.dh1 = g_topo_constants.dh1;
  if (!metrics_present(A.M, where)) return;
  const void* need[] = {T->xx, T->yy, T->zz, T->xy, T->xz, T->yz, T->r1, T->r2, T->r3,
                        T->r4, T->r5, T->r6, T->u1, T->v1, T->w1, T->lami, T->mui,
                        T->qpi, T->coeff, T->qsi, T->dcrjx, T->dcrjy, T->dcrjz};
  for (const void* x : need)
    if (!x) {
      awp_set_error(AWP_ERR_ARG, "%s: a field pointer is NULL", where);
      return;
    }
  if (texmode != TOPO_TEX_ARRAYS && (!rates || !tex)) {
    awp_set_error(AWP_ERR_ARG, "%s: the texture table applies to the two-pass update", where);
    return;
  }
  if ((texmode == TOPO_TEX_ARRAYS && (!T->vx1 || !T->vx2 || !T->ww || !T->wwo)) ||
      (texmode == TOPO_TEX_TABLE && !T->ww)) {
    awp_set_error(AWP_ERR_ARG, "%s: a relaxation-texture pointer is NULL", where);
    return;
  }
  // stress bounds (topography.c:377-420) shifted by ngsl+2 into array
  // indices (stress_attenuation.cu:34, 76-79)
  const int half = AWP_NGSL / 2, shift = AWP_NGSL + 2;
  const int left1 = half;
  const int right0 = T->nx - half;
  const int y0 = T->y_rank_f < 0 ? half : -half;
  const int y1 = T->y_rank_b < 0 ? T->ny - half : T->ny + half;
  G.bi = left1 + shift;
  G.ei = right0 + shift;
  G.bj = y0 + shift;
  G.ej = y1 + shift;
  if (G.ei <= G.bi || G.ej <= G.bj) return;
  hipStream_t st = T->stream_i;
  VelTiles V;
  topo_tiles(T->nz, VT_MAXW, &V);
  V.ichunk = awp_tuning().topo_str_ichunk;
  V.wsync = awp_tuning().topo_wsync;
  dim3 block(64, V.nseg * V.rj, 1);
  dim3 grid(V.nint + 1, awp_cdiv(G.ej - G.bj, V.rj), awp_cdiv(G.ei - G.bi, V.ichunk));
  const size_t lds = (size_t)2 * V.rj * ST_NC * V.ch * sizeof(float);
  if (!rates) {
    hipLaunchKernelGGL((topo_str_kernel<ST>), grid, block, lds, st, A, G, V);
    awp_check_launch(where);
    return;
  }
  // two passes: strain rates into rates, then the material and memory-
  // variable update streaming them back
  const long long rstride = (long long)G.sl * (T->nx + 4 + AWP_NGSL2);
  const int ni = G.ei - G.bi, nj = G.ej - G.bj;
  const size_t rlds = (size_t)2 * V.rj * 3 * (V.ch + 2 * VT_PAD) * sizeof(float);
  V.ichunk = topo_chunk(ni, (V.nint + 1) * nj * V.nseg, 24, awp_tuning().topo_rate_chunk);
  const dim3 gi(V.nint + 1, awp_cdiv(nj, V.rj), awp_cdiv(ni, V.ichunk));
  hipLaunchKernelGGL((topo_rates_kernel<ST, 0>), gi, block, rlds, st, A, G, V, rates, rstride);
  V.ichunk = topo_chunk(nj, (V.nint + 1) * ni * V.nseg, 24, awp_tuning().topo_rate_chunk);
  const dim3 gj(V.nint + 1, awp_cdiv(ni, V.rj), awp_cdiv(nj, V.ichunk));
  hipLaunchKernelGGL((topo_rates_kernel<ST, 1>), gj, block, rlds, st, A, G, V, rates, rstride);
  TopoQLaunch QL;
  QL.tile = awp_pick_tile(T->nz, false, 0, awp_tuning().kw);
  QL.nkt = QL.tile.nkt;
  QL.njt = awp_cdiv(nj, QL.tile.rows);
  int nic;
  awp_split_march(ni, QL.nkt * QL.njt, QL.tile.waves, awp_tuning().topo_q_ichunk, 10240, 16, &nic,
                  &QL.ichunk);
  QL.nblocks = QL.nkt * QL.njt * nic;
  const dim3 gq(QL.nblocks), bq(64 * QL.tile.waves);
  TopoTex TT = {};
  if (texmode != TOPO_TEX_ARRAYS) {
    for (int m = 0; m < 24; ++m) TT.t[m] = tex[m];
    // the stress region init_texture walks (mesh.c:1103-1137)
    TT.xls = 2 + AWP_NGSL;
    TT.yls = 2 + AWP_NGSL;
    TT.nj = T->ny;
    TT.nzt = T->nz;
  }
  if (texmode == TOPO_TEX_RULE)
    hipLaunchKernelGGL((topo_str_q_kernel<ST, TOPO_TEX_RULE>), gq, bq, 0, st, A, G,
                       rates, rstride, QL, TT);
  else if (texmode == TOPO_TEX_TABLE)
    hipLaunchKernelGGL((topo_str_q_kernel<ST, TOPO_TEX_TABLE>), gq, bq, 0, st, A, G,
                       rates, rstride, QL, TT);
  else
    hipLaunchKernelGGL((topo_str_q_kernel<ST, TOPO_TEX_ARRAYS>), gq, bq, 0, st, A, G,
                       rates, rstride, QL, TT);
  awp_check_launch(where);
}

bool neighbourless(int rank, const char* where) {
  if (rank >= 0) {
    awp_set_error(AWP_ERR_ARG,
                  "%s: a neighbouring rank (%d) needs the halo buffers of a multi-GPU run, "
                  "which this one-GPU library does not keep",
                  where, rank);
    return false;
  }
  return true;
}

}  // namespace

extern "C" {

void topo_set_constants(topo_t* T) {
  if (!T) {
    awp_set_error(AWP_ERR_ARG, "topo_set_constants: topo_t is NULL");
    return;
  }
  // set_constants(gridspacing, dth * gridspacing, ...) (stress_attenuation.cu:19-72)
  const float h = T->gridspacing;
  const float dt = T->dth * h;
  g_topo_constants.DT = dt;
  g_topo_constants.dth = dt / h;
  g_topo_constants.dh1 = (float)(1.0 / (double)h);
  g_topo_constants.set = 1;
}

void topo_velocity_interior_H(topo_t* T) {
  topo_velocity_launch<StF32>(T, WaveScales{}, "topo_velocity_interior_H");
}

void topo_velocity_front_H(topo_t* T) {
  if (T && T->use) neighbourless(T->y_rank_f, "topo_velocity_front_H");
}

void topo_velocity_back_H(topo_t* T) {
  if (T && T->use) neighbourless(T->y_rank_b, "topo_velocity_back_H");
}

void topo_stress_interior_H(topo_t* T) {
  topo_stress_launch<StF32>(T, WaveScales{}, "topo_stress_interior_H", nullptr);
}

void awp_topo_stress_interior_rates_H(topo_t* T, float* rates) {
  if (!rates) {
    awp_set_error(AWP_ERR_ARG, "awp_topo_stress_interior_rates_H: rates is NULL");
    return;
  }
  topo_stress_launch<StF32>(T, WaveScales{}, "awp_topo_stress_interior_rates_H", rates);
}

void awp_topo_stress_interior_tex_H(topo_t* T, float* rates, const float* tex, int rule) {
  const char* W = "awp_topo_stress_interior_tex_H";
  if (!rates || !tex) {
    awp_set_error(AWP_ERR_ARG, "%s: rates and tex must not be NULL", W);
    return;
  }
  topo_stress_launch<StF32>(T, WaveScales{}, W, rates, tex,
                            rule ? TOPO_TEX_RULE : TOPO_TEX_TABLE);
}

void topo_stress_left_H(topo_t* T) {
  if (T && T->use) neighbourless(T->x_rank_l, "topo_stress_left_H");
}

void topo_stress_right_H(topo_t* T) {
  if (T && T->use) neighbourless(T->x_rank_r, "topo_stress_right_H");
}

void awp_topo_velocity_s16(topo_t* T, int fmt, const float* scale) {
  WaveScales W;
  if (!awp_scales_from_host("awp_topo_velocity_s16", fmt, scale, &W)) return;
  if (fmt == AWP_FMT_BF16)
    topo_velocity_launch<StBF16>(T, W, "awp_topo_velocity_s16");
  else
    topo_velocity_launch<StF16>(T, W, "awp_topo_velocity_s16");
}

void awp_topo_stress_s16(topo_t* T, int fmt, const float* scale, float* rates) {
  WaveScales W;
  if (!awp_scales_from_host("awp_topo_stress_s16", fmt, scale, &W)) return;
  if (fmt == AWP_FMT_BF16)
    topo_stress_launch<StBF16>(T, W, "awp_topo_stress_s16", rates);
  else
    topo_stress_launch<StF16>(T, W, "awp_topo_stress_s16", rates);
}

void awp_topo_geom_custom(float* f, int nx, int ny, int nz, float h, hipStream_t St) {
  if (!f || nx < 1 || ny < 1 || nz < 3 || !(h > 0.0f)) {
    awp_set_error(AWP_ERR_ARG, "awp_topo_geom_custom: bad arguments");
    return;
  }
  const float normalize = (float)(1.0 / (double)h / (double)(nz - 2));
  const int frow = 2 * AWP_ALIGN + 2 * AWP_NGSL + ny + 4;
  dim3 grid(awp_cdiv(ny + 2 * AWP_NGSL, 64), nx + 2 * AWP_NGSL, 1);
  hipLaunchKernelGGL(geom_custom_kernel, grid, dim3(64), 0, St, f, nx, ny, frow, normalize);
  awp_check_launch("awp_topo_geom_custom");
}

void awp_topo_metrics_f(const f_grid_t* mf, int nx, int ny, float h, hipStream_t St) {
  if (!mf || nx < 1 || ny < 1 || !(h > 0.0f)) {
    awp_set_error(AWP_ERR_ARG, "awp_topo_metrics_f: bad arguments");
    return;
  }
  FPtrs F{mf->d_f, mf->d_f_1, mf->d_f_2, mf->d_f_c, mf->d_f1_1,
          mf->d_f1_2, mf->d_f1_c, mf->d_f2_1, mf->d_f2_2, mf->d_f2_c};
  const float* all[10] = {F.f, F.f_1, F.f_2, F.f_c, F.f1_1, F.f1_2, F.f1_c, F.f2_1, F.f2_2,
                          F.f2_c};
  for (const float* x : all)
    if (!x) {
      awp_set_error(AWP_ERR_ARG, "awp_topo_metrics_f: a metric array is NULL");
      return;
    }
  const int frow = 2 * AWP_ALIGN + 2 * AWP_NGSL + ny + 4;
  const float hi = (float)(1.0 / (double)h);  // f_grid_t.hi (metrics.c:24)
  dim3 grid(awp_cdiv(ny + 12, 64), nx + 12, 1);
  hipLaunchKernelGGL(metrics_interp_kernel, grid, dim3(64), 0, St, F, nx, ny, frow);
  if (!awp_check_launch("awp_topo_metrics_f")) return;
  hipLaunchKernelGGL(metrics_diff_kernel, grid, dim3(64), 0, St, F, nx, ny, frow, hi);
  awp_check_launch("awp_topo_metrics_f");
}

void awp_topo_geom_no_stretching(float* g, int nz, float h, hipStream_t St) {
  if (!g || nz < 18 || !(h > 0.0f)) {
    awp_set_error(AWP_ERR_ARG, "awp_topo_geom_no_stretching: bad arguments (nz >= 18)");
    return;
  }
  const float hi = (float)(1.0 / (double)h);   // g_grid_t.hi (metrics.c:211)
  const float hp = (float)(1.0 / (double)hi);  // the z grid spacing (metrics.c:335)
  hipLaunchKernelGGL(g_fill_kernel, dim3(awp_cdiv(nz, 64)), dim3(64), 0, St, g, nz, hp);
  awp_check_launch("awp_topo_geom_no_stretching");
}

void awp_topo_metrics_g(const g_grid_t* mg, int nz, float h, hipStream_t St) {
  if (!mg || !mg->d_g || !mg->d_g_c || !mg->d_g3 || !mg->d_g3_c || nz < 18 || !(h > 0.0f)) {
    awp_set_error(AWP_ERR_ARG, "awp_topo_metrics_g: bad arguments (nz >= 18, four arrays)");
    return;
  }
  const float hi = (float)(1.0 / (double)h);  // g_grid_t.hi (metrics.c:211)
  hipLaunchKernelGGL(metrics_g_kernel, dim3(1), dim3(256), 0, St, mg->d_g, mg->d_g_c, mg->d_g3,
                     mg->d_g3_c, nz, hi);
  awp_check_launch("awp_topo_metrics_g");
}

}  // extern "C"
