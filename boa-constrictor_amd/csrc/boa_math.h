// Device math shared by every kernel of the codec path.
//
// All code here is compiled with -ffp-contract=off: a multiply-add is fused
// only where __builtin_fmaf is written out.  The compress (chunk) and
// decompress (step) kernels call exactly these functions in the same order,
// which is what keeps their logits bit-identical (the decoder re-derives the
// encoder's integer CDFs from them).
//
// boa_expf / boa_logf are this project's own functions (not vendor libm):
//   exp: Cody-Waite reduction x = k ln2 + r with ln2 split in a float head and
//        tail, e^r by the degree-7 Taylor polynomial (Horner, fma), 2^k built
//        in the exponent field; x < -87 gives 0 so every result is normal.
//   log: y = 2^e m, m in [sqrt(1/2), sqrt(2)], log m = 2 atanh(s) with
//        s = (m-1)/(m+1), odd series to s^11.
// boa_repro_exp / tanh / gelu restate the reference's software activations
// (portability_solved_cpp/activations.hpp:33-117, device branch) operation
// for operation; the FF GELU of the reference uses them.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#define BOA_DEV __device__ __forceinline__

namespace boa {

BOA_DEV float u2f(uint32_t u) { return __uint_as_float(u); }
BOA_DEV uint32_t f2u(float f) { return __float_as_uint(f); }

// bfloat16 storage (uint16_t): the upper half of a float32, rounded to
// nearest even by gfx950's v_cvt_pk_bf16_f32; a NaN stays a quiet NaN.
BOA_DEV uint16_t f32_to_bf16(float x) { return __builtin_bit_cast(uint16_t, (__bf16)x); }
BOA_DEV float bf16_to_f32(uint16_t h) { return u2f((uint32_t)h << 16); }
BOA_DEV float bf16r(float x) { return bf16_to_f32(f32_to_bf16(x)); }

// activation storage: fp32 or bf16
BOA_DEV float ldv(const float* p) { return *p; }
BOA_DEV float ldv(const uint16_t* p) { return bf16_to_f32(*p); }
BOA_DEV void stv(float* p, float v) { *p = v; }
BOA_DEV void stv(uint16_t* p, float v) { *p = f32_to_bf16(v); }

// What an fp32 element costs on gfx950 (a wave64 instruction's issue on one
// SIMD, measured with independent chains): add, mul and fma on VGPRs,
// literals or inline constants, integer add and the bit operations about 2.4
// cycles; anything with an SGPR operand, min / max / med3, rounding,
// conversions, shifts, ldexp, compares, selects and the div_ helpers 4.2; the
// transcendentals 8.2.  fp32 MFMAs issue no faster than that and not beside
// it (eight fma and one 16x16x4 MFMA take 22 + 34 cycles), so the functions
// below prefer adds and fmas to the instructions named for a job:
//   - rint(y), |y| < 2^22, is (y + 1.5 2^23) - 1.5 2^23, and the sum's low
//     bits are the integer itself: p 2^k is an exponent-field add
//     (v_lshl_add) instead of rndne + cvt + ldexp;
//   - a division whose operands and quotient stay in the normal range needs
//     no scaling and no fix-up (div_normal);
//   - one comparison of the whole wave picks the form for ordinary arguments
//     (no clamps, no selects) or the general one (wave_ordinary).
// The results are those of the general forms for every float.

// RINT_MAGIC + y: rint(y) in the low mantissa bits for |y| < 2^22.
constexpr float RINT_MAGIC = 12582912.0f;
// p 2^k for k = rint_sum - RINT_MAGIC; p, p 2^k normal (or p 2^k = 2^128 = inf).
BOA_DEV float scale_rint(float p, float rint_sum) { return u2f(f2u(p) + (f2u(rint_sum) << 23)); }

// n / d, correctly rounded, for normal d with a normal reciprocal, n / d zero
// or normal, and n zero or |n| >= 2^-100 (so that the residuals n - d q do not
// underflow): Newton's step on the reciprocal, then two residual corrections
// of the quotient (Markstein).  8 instructions, 27
// cycles, against 12 and about 45 for the scaled division.
BOA_DEV float div_normal(float n, float d) {
  float y = __builtin_amdgcn_rcpf(d);
  y = __builtin_fmaf(__builtin_fmaf(-d, y, 1.0f), y, y);
  float q = n * y;
  q = __builtin_fmaf(__builtin_fmaf(-d, q, n), y, q);
  return __builtin_fmaf(__builtin_fmaf(-d, q, n), y, q);
}

// whether every active lane's predicate holds (a scalar branch, no divergence)
BOA_DEV bool wave_ordinary(bool p) {
  return __builtin_expect(__builtin_amdgcn_ballot_w64(!p) == 0, 1);
}

// e^x and log(y): expf_ is branch-free (the arithmetic runs on a clamped
// argument and selects give the special values), expf_br returns early on
// them; the results are the same for every input.

// e^x for x in [-87, 88.7228...), where it is finite
BOA_DEV float exp_core(float x) {
  const float LOG2E = 1.44269504088896340736f;
  const float LN2_HI = 0.693147182464599609375f;
  const float LN2_LO = -1.904654323148236e-09f;
  const float km = x * LOG2E + RINT_MAGIC;
  const float kf = km - RINT_MAGIC;
  float r = __builtin_fmaf(-kf, LN2_HI, x);
  r = __builtin_fmaf(-kf, LN2_LO, r);
  float p = 1.98412698412698412698e-4f;
  p = __builtin_fmaf(p, r, 1.38888888888888888889e-3f);
  p = __builtin_fmaf(p, r, 8.33333333333333333333e-3f);
  p = __builtin_fmaf(p, r, 4.16666666666666666667e-2f);
  p = __builtin_fmaf(p, r, 1.66666666666666666667e-1f);
  p = __builtin_fmaf(p, r, 0.5f);
  p = __builtin_fmaf(p, r, 1.0f);
  p = __builtin_fmaf(p, r, 1.0f);
  return scale_rint(p, km);
}

BOA_DEV float expf_(float x) {
  float res = exp_core(__builtin_fminf(__builtin_fmaxf(x, -87.0f), 88.72283935546875f));
  res = x < -87.0f ? 0.0f : res;
  res = x >= 88.72283935546875f ? __builtin_huge_valf() : res;
  return x != x ? x : res;
}

// 2^t for t <= 0, the exponentials whose argument is never positive: the
// selective scan's decay exp(-exp(A_log) dt), taken in base 2 (the weights
// hold na2 = -exp(A_log) * log2(e), two fp32 roundings done once at load,
// and the scan takes 2^t of t = na2 * dt), and the CDF's exp(l - max),
// taken as 2^((l - max) log2(e)).  t is clamped into
// [-126, 0] (fmaxf turns a NaN into -126), split as k + r with k = rint(t)
// and r = t - k in [-1/2, 1/2] (exact); 2^r comes from a degree-6
// polynomial with 2^0 = 1 exact, fitted to the relative error of 2^r on
// [-1/2, 1/2] (under one ulp with fp32 fma evaluation), and 2^k is added to
// the exponent field.  The least result is 2^-126: no subnormal is produced.
// exp2_neg_core: t already in [-126, 0] (29 cycles an element, against 37
// with the clamp, rndne, cvt and ldexp).
BOA_DEV float exp2_neg_core(float s) {
  const float km = s + RINT_MAGIC;
  const float r = s - (km - RINT_MAGIC);
  float p = 0x1.41fbbap-13f;
  p = __builtin_fmaf(p, r, 0x1.5f3e54p-10f);
  p = __builtin_fmaf(p, r, 0x1.3b2d4cp-7f);
  p = __builtin_fmaf(p, r, 0x1.c6aee8p-5f);
  p = __builtin_fmaf(p, r, 0x1.ebfbdcp-3f);
  p = __builtin_fmaf(p, r, 0x1.62e430p-1f);
  p = __builtin_fmaf(p, r, 1.0f);
  return scale_rint(p, km);
}
BOA_DEV float exp2_neg(float t) {
  return exp2_neg_core(__builtin_fminf(__builtin_fmaxf(t, -126.0f), 0.0f));
}

BOA_DEV float expf_br(float x) {
  if (x != x) return x;
  if (x >= 88.72283935546875f) return __builtin_huge_valf();
  if (x < -87.0f) return 0.0f;
  return exp_core(x);
}

// log(y) for y in [1, 2^127): y = 2^e m with m in (sqrt(1/2), sqrt(2)]
BOA_DEV float log_core(float y) {
  const uint32_t above = f2u(y) - 0x3F3504F4u;  // from the least float over sqrt(1/2)
  const int e = (int)above >> 23;
  const float m = u2f(f2u(y) - (above & 0xFF800000u));
  const float s = div_normal(m - 1.0f, m + 1.0f);
  const float s2 = s * s;
  float p = 0.0909090909090909090909f;
  p = __builtin_fmaf(p, s2, 0.111111111111111111111f);
  p = __builtin_fmaf(p, s2, 0.142857142857142857143f);
  p = __builtin_fmaf(p, s2, 0.2f);
  p = __builtin_fmaf(p, s2, 0.333333333333333333333f);
  const float two_s = s + s;
  const float lm = __builtin_fmaf(two_s * s2, p, two_s);
  const float LN2_HI = 0.693147182464599609375f;
  const float LN2_LO = -1.904654323148236e-09f;
  const float ef = (float)e;
  return __builtin_fmaf(ef, LN2_HI, __builtin_fmaf(ef, LN2_LO, lm));
}

// Forms of the transcendental activations.  MATH_BF and MATH_BR give
// identical results (branch-free vs early-return special cases; the
// oracle's functions).  MATH_HW uses the hardware exp2/log2/reciprocal
// (v_exp_f32, v_log_f32, v_rcp_f32, about 1 ulp): the bf16 precision runs on
// it in compress and decode alike, so its two passes still agree bit for
// bit while its logits are compared with the oracle within the bf16
// tolerance.
enum { MATH_BF = 0, MATH_BR = 1, MATH_HW = 2 };

BOA_DEV float hw_exp(float x) { return __builtin_amdgcn_exp2f(x * 1.44269504088896340736f); }
BOA_DEV float hw_log(float x) { return __builtin_amdgcn_logf(x) * 0.69314718055994530942f; }
BOA_DEV float hw_rcp(float x) { return __builtin_amdgcn_rcpf(x); }

template <int M>
BOA_DEV float exp_sel(float x) { return M == MATH_HW ? hw_exp(x) : M == MATH_BR ? expf_br(x) : expf_(x); }

// |x| up to which sigmoid_core and softplus_core hold: e^87 < 2^126, so
// 1 + e^x and its reciprocal are normal
constexpr float ORDINARY = 87.0f;
// 1 / (1 + e^-x) and log(1 + e^x) for |x| <= ORDINARY
BOA_DEV float sigmoid_core(float x) { return div_normal(1.0f, 1.0f + exp_core(-x)); }
BOA_DEV float softplus_core(float x) { return log_core(1.0f + exp_core(x)); }
// ... and for every x: e^x = 0 below -87 leaves 1 + 0, whose log is 0; above
// 88.72 it is inf, whose log is inf and reciprocal 0
template <int M>
BOA_DEV float sigmoid_any(float x) { return 1.0f / (1.0f + exp_sel<M>(-x)); }
template <int M>
BOA_DEV float softplus_any(float x) {
  const float c = log_core(1.0f + exp_core(__builtin_fminf(__builtin_fmaxf(x, -87.0f), 87.0f)));
  if (__builtin_fabsf(x) <= ORDINARY) return c;
  const float y = 1.0f + exp_sel<M>(x);  // 1, [2^125, 2^128), inf or NaN
  return y < __builtin_huge_valf() ? log_core(y) : y;
}

// activations.hpp:33-84 (device branch) for x in [-20, 20], the arguments
// that tanh's saturation leaves
BOA_DEV float repro_exp_core(float x) {
  const float kf = __builtin_floorf(x * 1.44269504088896340736f + 0.5f);
  float r = x + (-(kf * 0.69314718055994530942f));
  float t = 0.008333333333f + r * 0.001388888889f;
  t = 0.041666666667f + r * t;
  t = 0.166666666667f + r * t;
  t = 0.5f + r * t;
  t = 1.0f + r * t;
  t = 1.0f + r * t;
  return scale_rint(t, kf + RINT_MAGIC);
}

// activations.hpp:87-98: (e^2x - 1) / (e^2x + 1), and +-1 where |x| > 10.
// The quotient at +-10 is +-1 exactly (e^20 +- 1 and e^-20 +- 1 round to
// e^20 and to +-1), so clamping x to [-10, 10] gives the saturation without
// selects; a NaN is left to the caller's product with x.  In hardware
// arithmetic 1 - 2 / (e^2x + 1) saturates by itself.
template <int M>
BOA_DEV float repro_tanh(float x) {
  if (M == MATH_HW) return __builtin_fmaf(-2.0f, hw_rcp(hw_exp(2.0f * x) + 1.0f), 1.0f);
  const float e2x = repro_exp_core(2.0f * __builtin_fminf(__builtin_fmaxf(x, -10.0f), 10.0f));
  return div_normal(e2x + -1.0f, e2x + 1.0f);
}

// activations.hpp:105-117 (tanh GELU used by the FF epilogue).  fp32 on
// gfx950: about 106 cycles an element against 160 with the selects and the
// scaled division.
template <int M = MATH_BF>
BOA_DEV float gelu(float x) {
  float cube = (x * x) * x;
  float inner = 0.79788456080286535588f * (x + 0.044715f * cube);
  float th = repro_tanh<M>(inner);
  return 0.5f * (x * (1.0f + th));
}

// 1 / (1 + exp(-x)) of the gate and SiLU
template <int M = MATH_BF>
BOA_DEV float sigmoid(float x) {
  if (M == MATH_HW) return hw_rcp(1.0f + hw_exp(-x));
  return wave_ordinary(__builtin_fabsf(x) <= ORDINARY) ? sigmoid_core(x) : sigmoid_any<M>(x);
}

// SiLU in the form v * (1 / (1 + exp(-v))) (mamba_kernels.cu:188-189)
template <int M = MATH_BF>
BOA_DEV float silu(float x) { return x * sigmoid<M>(x); }

// ... of N values at once, one form for all of them: one branch, their chains
// side by side
template <int M, int N>
BOA_DEV void silu_each(float (&v)[N]) {
  if constexpr (M == MATH_HW) {
#pragma unroll
    for (int k = 0; k < N; ++k) v[k] = silu<M>(v[k]);
  } else {
    bool ordinary = true;
#pragma unroll
    for (int k = 0; k < N; ++k) ordinary &= __builtin_fabsf(v[k]) <= ORDINARY;
    if (wave_ordinary(ordinary)) {
#pragma unroll
      for (int k = 0; k < N; ++k) v[k] = v[k] * sigmoid_core(v[k]);
    } else {
#pragma unroll
      for (int k = 0; k < N; ++k) v[k] = v[k] * sigmoid_any<M>(v[k]);
    }
  }
}

// unthresholded softplus log(1 + exp(x)) (inference_kernels.cu:376-382)
template <int M = MATH_BF>
BOA_DEV float softplus(float x) {
  if (M == MATH_HW) return hw_log(1.0f + hw_exp(x));
  return wave_ordinary(__builtin_fabsf(x) <= ORDINARY) ? softplus_core(x) : softplus_any<M>(x);
}

// 2^t for t <= 0 (see exp2_neg) in the chosen form
template <int M>
BOA_DEV float exp2_neg_sel(float t) {
  return M == MATH_HW ? __builtin_amdgcn_exp2f(t) : exp2_neg(t);
}

// the scan's base-2 decay coefficient from A_log (see exp2_neg)
BOA_DEV float scan_na2(float a_log) { return -expf_(a_log) * 1.44269504088896340736f; }

}  // namespace boa
