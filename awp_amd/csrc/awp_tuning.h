// Launch-shape knobs shared by the launchers (set with awp_set_tuning).
#pragma once

struct AwpTuning {
  int vel_bj;       // waves per velocity workgroup (0: awp_pick_tile)
  int str_bj;       // waves per stress workgroup (0: awp_pick_tile)
  int vel_target_wgs;  // velocity: workgroups to aim for when splitting the i march
  int str_target_wgs;  // stress: same
  int vel_ichunk;   // >0 forces the velocity i-chunk length
  int str_ichunk;   // >0 forces the stress i-chunk length
  int xcd_remap;    // 1: XCD-aware tile order, 0: plain order
  int kalign;       // 1: start k tiles on a 32-float (128 B) line boundary
  int topo_vel_ichunk;  // planes per march of the curvilinear velocity kernel (0: topo_chunk)
  int topo_str_ichunk;  // same, one-pass curvilinear stress kernel
  int topo_q_ichunk;    // same, second pass of the two-pass update (0: awp_split_march)
  int step_ichunk;      // >0 forces the i-chunk length of the fused step (awp_step)
  int step_target_wgs;  // fused step: workgroups to aim for when splitting the i march
  int vel_jfast;        // 1: j tiles fastest in the block order (velocity)
  int str_jfast;        // same, stress
  int step_jfast;       // same, fused step
  int adj_jgroup;       // adjoint kernels' block order: 0 plane by plane, else j tiles per group
  int kw;               // k-run width of the Cartesian kernels: 0 by the idle-lane rules, 32, 64
  int topo_nseg;        // curvilinear kernels: waves per k chunk at most (1: one-wave segments)
  int topo_wsync;       // curvilinear kernels: 1 wave-scope LDS sync where a wave reads only its own
  int topo_rate_chunk;  // > 0 forces the planes per march of the strain-rate launches
  int topo_rj;          // curvilinear kernels: > 0 forces the j rows per workgroup
};

AwpTuning& awp_tuning();

// Chunks of a march over ni planes whose tiling gives nkj workgroups of `waves`
// waves per chunk, for the Cartesian kernels and the second curvilinear stress
// pass: 4 (or `most`, if less) to `most` planes towards `target` workgroups of 4 waves (10240 = 40
// per CU).  Longer chunks re-read fewer planes at their ends but leave the last
// round of workgroups nearly empty.  most = 16 for the stress updates: at
// 243x187x101 chunks of 4 against 16 planes took the stress update (per-cell
// texture) 194 against 216 us, at 400x300x200 8 against 32 took 860 against 938
// us; at 512x512x256 16 and longer are level (1.99 ms).  A grid too small for
// one round of 1280 workgroups (5 per CU) at 4 planes takes fewer.
static inline void awp_split_march(int ni, int nkj, int waves, int forced, int target, int most,
                                   int* nic, int* ichunk) {
  const long long planes = (long long)ni * nkj * waves / 4;
  long long c = planes / target;
  if (c < 4) c = 4;
  if (c > most) c = most;
  if (c > planes / 1280) c = planes / 1280;
  if (forced > 0) c = forced;
  if (c < 1) c = 1;
  *ichunk = (int)c;
  *nic = (ni + (int)c - 1) / (int)c;
}

// Number of i-chunks and chunk length for a march over ni planes when the
// (k, j) tiling gives nkj workgroups per chunk.
static inline void awp_split_i(int ni, int nkj, int forced, int target, int* nic, int* ichunk) {
  int c;
  if (forced > 0) {
    c = forced;
  } else {
    int want = (target + nkj - 1) / nkj;
    if (want < 1) want = 1;
    if (want > ni) want = ni;
    c = (ni + want - 1) / want;
  }
  if (c < 1) c = 1;
  *ichunk = c;
  *nic = (ni + c - 1) / c;
}
