// Binary32 division by an explicit reciprocal, and the branch tests of the
// coarse-grained Q weights without a division.
//
// hipcc lowers a binary32 a / b to 11 VALU instructions and two writes of
// the mode register (it turns binary32 denormals on around its refinement),
// and a binary64 one to about 14.  One cell of the stress update divides
// fifteen times: 170 of its 530 VALU instructions.  Here:
//   * the reciprocal is v_rcp_f32 (error below 1 ulp) and one Newton step in
//     fused arithmetic, which gives the correctly rounded 1/b (not by a general
//     theorem: by what the instruction returns, which the tests check for all
//     2^23 significands);
//   * a quotient is a*y corrected once by its exact residual,
//     q = fma(fma(-a*y, b, a), y, a*y), which with y = RN(1/b) is the
//     correctly rounded a/b (P. W. Markstein, "Computation of elementary
//     functions on the IBM RISC System/6000 processor", IBM J. Res. Dev.
//     34(1), 1990);
//   * v_div_fixup_f32 puts the IEEE results in place for zeros, infinities
//     and NaN.
// So the quotient's bits are those of a / b wherever a, b, 1/b and a/b are
// normal numbers whose residual (2^-24 a) is one too: |a| > 2^-100 or a = 0,
// 2^-125 < |b| < 2^125.  For smaller a the residual is flushed and the quotient
// is a*y, within 2 ulps of a / b.  Only the plasticity kernels divide fields:
// stresses (Pa, 2^-100 is 8e-31) by 3, by the root of their second invariant
// and by a modulus.  Values that small take part in the results through
// squares, which flush to zero, or are added to terms 2^24 times larger.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

// 1/b, correctly rounded for normal b and 1/b; NaN for b = 0, inf (the
// callers' fixups overwrite it).
__device__ __forceinline__ float awp_rcp(float b) {
  const float y = __builtin_amdgcn_rcpf(b);
  return __builtin_fmaf(__builtin_fmaf(-b, y, 1.0f), y, y);
}

// a / b with y = awp_rcp(b).
__device__ __forceinline__ float awp_div_by(float a, float b, float y) {
  const float q = a * y;
  return __builtin_amdgcn_div_fixupf(__builtin_fmaf(__builtin_fmaf(-q, b, a), y, q), b, a);
}

__device__ __forceinline__ float awp_div(float a, float b) { return awp_div_by(a, b, awp_rcp(b)); }

// c / b for a power of two c: scaling by c is exact.
__device__ __forceinline__ float awp_pow2_div(float c, float b) {
  return __builtin_amdgcn_div_fixupf(c * awp_rcp(b), b, c);
}

// 1. / (2. * q) <= 200.0 in binary64 (the production Q weights), and
// 1.0f / (2.0f * q) <= 200.0f in binary32, as one integer comparison: the
// quotient falls with q > 0, so the test is q >= the smallest binary32 q that
// passes (binary64: the binary32 above 0.0025; binary32: 0.0025 itself,
// whose quotient rounds to 200).  Negative q pass, as their quotients do;
// -0 and NaN pass here and only choose between two zeros or two NaN.
__device__ __forceinline__ bool awp_q_low64(float q) {
  return __builtin_bit_cast(uint32_t, q) >= 0x3b23d70bu;
}
__device__ __forceinline__ bool awp_q_low32(float q) {
  return __builtin_bit_cast(uint32_t, q) >= 0x3b23d70au;
}

// Coarse-grained Q weights, y = awp_rcp(wwo).  Both branches are cheaper than
// a divergent branch around either.
// The production update's (kernel.cu:978-1045): binary64 test and quadratic.
__device__ __forceinline__ float awp_qw_prod(float q, float ca, float cb, float wwo, float y) {
  const double t = 2. * (double)q;
  const float quad = (float)((double)ca * t * t + (double)cb * t);
  return awp_div_by(awp_q_low64(q) ? quad : 2.0f * wwo * q, wwo, y);
}

// dstrqc_new's (kernel.cu:505-604) and the curvilinear update's: binary32
// test; qpa keeps a binary64 quadratic (dbl), the others are binary32.
__device__ __forceinline__ float awp_qw_new(float q, float ca, float cb, float wwo, float y,
                                            bool dbl) {
  float quad;
  if (dbl) {
    const double t = 2. * (double)q;
    quad = (float)((double)ca * t * t + (double)cb * t);
  } else {
    quad = ca * (2.0f * q) * (2.0f * q) + cb * (2.0f * q);
  }
  return awp_div_by(awp_q_low32(q) ? quad : 2.0f * wwo * q, wwo, y);
}
