// Shared definitions for the gfx950 AWP-ODC kernels.
//
// Memory layout (reference src/awp/kernel.cu:87-94, src/awp/grid.c:14-38):
// every 3-D field is one flat float array with k (z) fastest, then j, then i:
//   p = i*slice + j*yline + k,  yline = nzt + 2*align,
//   slice = (nyt + 4 + 2*ngsl) * yline.
// Interior: i in [2+ngsl, nxt+ngsl+1], j in [2+ngsl, nyt+ngsl+1],
// k in [align, nzt+align-1]; k = nzt+align-1 is the free surface.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#define AWP_NGSL 8        // include/awp/pmcl3d_cons.h:22
#define AWP_NGSL2 16      // include/awp/pmcl3d_cons.h:23
#define AWP_ALIGN 32      // include/awp/pmcl3d_cons.h:16
#define AWP_MAXGRIDS 10   // include/awp/pmcl3d_cons.h:77
#define AWP_NXCD 8        // MI355X: 8 accelerator complex dies, each with its own L2

// Per-grid scalars, derived exactly as SetDeviceConstValue derives them
// (src/awp/kernel.cu:68-117).  They travel to kernels by value (kernarg
// segment -> scalar registers) instead of through __constant__ symbols.
struct AwpGrid {
  float c1, c2, dth, dh1, DT, DH;
  int nxt, nyt, nzt;
  int yline;      // nzt + 2*align
  long long slice;  // (nyt+4+ngsl2) * yline
};

// Plasticity constants (SetDeviceConstValue's fmajor/fminor/Rz/RzT).
struct AwpPlastConst {
  float fmajor, fminor;
  float Rz[9], RzT[9];
};

// Host-side state filled by SetDeviceConstValue; process-global like the
// reference's __constant__ block (not re-entrant, at most AWP_MAXGRIDS grids).
struct AwpState {
  int ngrids;
  int initialised;
  AwpGrid grid[AWP_MAXGRIDS];
  AwpPlastConst plast;
};

AwpState& awp_state();

// Error reporting.  The reference's launchers return void and either print or
// exit (pmcl3d_cons.h:43-53, kernel.cu:1233-1235).  These record the first
// error since the last awp_clear_error() and print it to stderr; the Python
// layer raises on it.
void awp_set_error(int code, const char* fmt, ...);
bool awp_check_launch(const char* where);
bool awp_grid_ok(int d_i, const char* where);

// XCD-aware tile order.  The hardware hands workgroup b to XCD (b % 8); this
// renumbers workgroups so that each XCD receives one contiguous run of logical
// tiles, which keeps the j/k halo lines neighbouring tiles share inside one
// L2.  The map is a bijection on [0, nblocks).  Applied to the blocks of one
// i-chunk of a march at a time, it keeps the XCDs in the same few planes, each
// with a run of the chunk's tiles (where the chunk's size is no multiple of 8,
// the runs move on by that remainder from XCD to XCD with every chunk).
__host__ __device__ __forceinline__ int awp_xcd_remap(int b, int nblocks) {
  const int q = nblocks / AWP_NXCD, r = nblocks % AWP_NXCD;
  const int x = b % AWP_NXCD, s = b / AWP_NXCD;
  return x * q + (x < r ? x : r) + s;
}

static inline int awp_cdiv(int a, int b) { return (a + b - 1) / b; }

// (k, j) tile of the marching Cartesian kernels: a workgroup of `waves` waves
// covers `rows` j rows of `width` consecutive k each, lane t being row
// t / width and level t % width, `nkt` tiles down a column of n levels.
//   n <= 32: rows of 32 levels, two per wave (4 waves).  A column of n levels
//     would keep n of a wave's 64 lanes busy: 256x256x32 velocity 40.6 against
//     34.4 us, stress 99.5 against 74.9; in bfloat16 33.0 / 26.3 and 78.4 / 55.6;
//   64 < n <= 96 in 16-bit storage: likewise, three runs a row.  One row of 72 to
//     96 levels idles 32 to 56 lanes of 128, and a seam costs less where a line
//     holds 64 cells: bfloat16 150x130x90 velocity 24.8 / 22.9 us, stress 50.9 /
//     47.8; 512x512x96 289 / 257 and 675 / 652 (binary32 288x288x96 119 / 138
//     and 254 / 239, so rows there);
//   n <= 64, n a multiple of 64, n > 256: rows of 64 levels, one per wave
//     (4 waves), so a wave's accesses are whole 128-byte lines;
//   else: one row of all n levels, ceil(n / 64) waves.  Cut into runs, such a
//     column has seams inside it, and where nzt + 64 is no multiple of 32
//     every row starts inside a line: the lines at a seam are fetched by two
//     workgroups and written in two parts.  At 400x300x200 runs of 50 levels
//     fetched 2.51 GB and wrote 1.31 GB per stress update for 1.82 and 1.15
//     algorithmic; one row per workgroup took it from 899 to 829 us and the
//     velocity update from 393 to 340, idle lanes included (300x300xn: within
//     2 % of the best of 30 shapes for n = 101 .. 230).
// waves, width: forced by the tuning unless 0.
struct AwpTile {
  int width, rows, waves, nkt, mul;  // mul: t / width = t * mul >> 20 for t < 1024
};
static inline AwpTile awp_pick_tile(int n, bool bits16, int waves, int width) {
  AwpTile t;
  const bool run32 = n <= 32 || (bits16 && n > 64 && n <= 96);
  const bool row = !run32 && n > 64 && n <= 256 && n % 64 != 0;
  t.waves = waves > 0 ? waves : row && width <= 0 ? awp_cdiv(n, 64) : 4;
  t.width = width > 0 ? width : row ? n : run32 ? 32 : 64;
  if (t.width > 64 * t.waves) t.width = 64;
  t.rows = 64 * t.waves / t.width;
  t.nkt = awp_cdiv(n, t.width);
  t.mul = ((1 << 20) + t.width - 1) / t.width;
  return t;
}

// The tile of the plasticity kernels, which spend as many cycles on
// arithmetic as on memory (binary64 sine, cosine and exponential), so that idle
// lanes cost more than seams inside a column.
//   n <= 128: whole columns, in the workgroup of 1, 2, 3, 4 or 8 waves that
//     leaves the fewest lanes idle, the smaller one among equals (n = 48: 3
//     waves of 4 rows, all lanes; 64-level rows keep 75 %).  Not 5, 6 or 7:
//     drprecpc_calc holds 100 VGPRs, four waves per SIMD, which such workgroups
//     cannot fill evenly (256x256x96 calc 101 us with 3 waves, 158 with 5);
//   else: runs of 64 levels, or of 32 where those leave fewer lanes idle, 4
//     waves.  Whole columns (equal parts of them above 256) took 247 against 176
//     us at 256x256x150, 265 / 225 at 256x256x200 and 462 / 312 at 256x256x300.
static inline AwpTile awp_pick_full_tile(int n, int width) {
  AwpTile t;
  t.waves = 4;
  if (width > 0) {
    t.width = width;
  } else if (n > 128) {
    t.width = awp_cdiv(n, 32) * 32 < awp_cdiv(n, 64) * 64 ? 32 : 64;
  } else {
    t.width = n;
    float best = 0.0f;
    for (int w : {1, 2, 3, 4, 8}) {
      const float use = (float)(64 * w / n * n) / (float)(64 * w);
      if (use > best + 0.001f) {
        best = use;
        t.waves = w;
      }
    }
  }
  t.rows = 64 * t.waves / t.width;
  t.nkt = awp_cdiv(n, t.width);
  t.mul = ((1 << 20) + t.width - 1) / t.width;
  return t;
}

// The reference's (float)(c / (double)x) for binary32 c and x.  Rounding the
// binary64 quotient to binary32 gives the correctly rounded binary32 quotient:
// double rounding is innocuous when the wider format has at least 2p+2
// significand bits, and 53 >= 2*24+2 (S. A. Figueroa, "When is double rounding
// innocuous?", ACM SIGNUM Newsletter 30(3), 1995).  So one binary32 division
// (correctly rounded: hipcc's default) gives the same bits without binary64
// arithmetic.  A quotient in the subnormal range flushes to zero either way in
// this build.
__device__ __forceinline__ float awp_quot(float c, float x) { return c / x; }

// (k tile, j tile, i chunk) of logical block b: k tiles fastest, or with
// jfast the j tiles fastest, so that consecutive blocks (one XCD's L2 after
// awp_xcd_remap) are j neighbours and share their halo rows.
__device__ __forceinline__ void awp_tile3(int b, int nkt, int njt, int jfast, int& kt, int& jt,
                                          int& ic) {
  if (jfast) {
    jt = b % njt;
    kt = (b / njt) % nkt;
  } else {
    kt = b % nkt;
    jt = (b / nkt) % njt;
  }
  ic = b / (nkt * njt);
}

// Loads and stores through a wave-uniform row pointer and a per-lane 32-bit
// byte offset.  With one wave per j row the row pointer lives in scalar
// registers and every access of a row lowers to
// global_load/store v, v_koff, s[base:base+1]: one lane-offset VGPR shared
// by all fields instead of a 64-bit address pair per access.
__device__ __forceinline__ float awp_ld(const float* row, unsigned kbyte) {
  return *reinterpret_cast<const float*>(reinterpret_cast<const char*>(row) + kbyte);
}
__device__ __forceinline__ int awp_ldi(const int* row, unsigned kbyte) {
  return *reinterpret_cast<const int*>(reinterpret_cast<const char*>(row) + kbyte);
}
__device__ __forceinline__ void awp_st(float* row, unsigned kbyte, float v) {
  *reinterpret_cast<float*>(reinterpret_cast<char*>(row) + kbyte) = v;
}

