// The kernels' math functions (boa_math.h) against their plain forms -- ldexp
// for 2^k, the compiler's division, every special case by comparison -- over
// all 2^32 floats, on the GPU.  The plain forms are the CPU oracle's,
// operation for operation; plain() gives their values to compare with it.
#include <cstdint>

#include "../boa-constrictor_amd/csrc/boa_math.h"

namespace {
using namespace boa;

__device__ float plain_exp(float x) {
  if (x != x) return x;
  if (x > 88.72283935546875f) return __builtin_huge_valf();
  if (x < -87.0f) return 0.0f;
  const float kf = __builtin_rintf(x * 1.44269504088896340736f);
  float r = __builtin_fmaf(-kf, 0.693147182464599609375f, x);
  r = __builtin_fmaf(-kf, -1.904654323148236e-09f, r);
  float p = 1.98412698412698412698e-4f;
  p = __builtin_fmaf(p, r, 1.38888888888888888889e-3f);
  p = __builtin_fmaf(p, r, 8.33333333333333333333e-3f);
  p = __builtin_fmaf(p, r, 4.16666666666666666667e-2f);
  p = __builtin_fmaf(p, r, 1.66666666666666666667e-1f);
  p = __builtin_fmaf(p, r, 0.5f);
  p = __builtin_fmaf(p, r, 1.0f);
  p = __builtin_fmaf(p, r, 1.0f);
  return __builtin_ldexpf(p, (int)kf);
}

__device__ float plain_exp2_neg(float t) {
  const float s = __builtin_fminf(__builtin_fmaxf(t, -126.0f), 0.0f);
  const float k = __builtin_rintf(s), r = s - k;
  float p = 0x1.41fbbap-13f;
  p = __builtin_fmaf(p, r, 0x1.5f3e54p-10f);
  p = __builtin_fmaf(p, r, 0x1.3b2d4cp-7f);
  p = __builtin_fmaf(p, r, 0x1.c6aee8p-5f);
  p = __builtin_fmaf(p, r, 0x1.ebfbdcp-3f);
  p = __builtin_fmaf(p, r, 0x1.62e430p-1f);
  p = __builtin_fmaf(p, r, 1.0f);
  return __builtin_ldexpf(p, (int)k);
}

__device__ float plain_log(float y) {  // y >= 1, inf or NaN
  if (y != y || y == __builtin_huge_valf()) return y;
  const uint32_t u = f2u(y);
  int e = (int)(u >> 23) - 127;
  float m = u2f((u & 0x007FFFFFu) | 0x3F800000u);
  if (m > 1.41421353816986083984375f) {
    m = m * 0.5f;
    e += 1;
  }
  const float s = (m - 1.0f) / (m + 1.0f);
  const float s2 = s * s;
  float p = 0.0909090909090909090909f;
  p = __builtin_fmaf(p, s2, 0.111111111111111111111f);
  p = __builtin_fmaf(p, s2, 0.142857142857142857143f);
  p = __builtin_fmaf(p, s2, 0.2f);
  p = __builtin_fmaf(p, s2, 0.333333333333333333333f);
  const float two_s = s + s, lm = __builtin_fmaf(two_s * s2, p, two_s), ef = (float)e;
  return __builtin_fmaf(ef, 0.693147182464599609375f,
                        __builtin_fmaf(ef, -1.904654323148236e-09f, lm));
}

__device__ float plain_repro_exp(float x) {
  if (x <= -88.0f) return 0.0f;
  if (x >= 88.0f) x = 88.0f;
  const float kf = __builtin_floorf(x * 1.44269504088896340736f + 0.5f);
  const float r = x + (-(kf * 0.69314718055994530942f));
  float t = 0.008333333333f + r * 0.001388888889f;
  t = 0.041666666667f + r * t;
  t = 0.166666666667f + r * t;
  t = 0.5f + r * t;
  t = 1.0f + r * t;
  t = 1.0f + r * t;
  return t * u2f((uint32_t)(((int)kf + 127) << 23));
}

__device__ float plain_gelu(float x, bool hw) {
  const float inner = 0.79788456080286535588f * (x + 0.044715f * ((x * x) * x));
  float th;
  if (__builtin_fabsf(inner) > 10.0f) {
    th = inner > 0.0f ? 1.0f : -1.0f;
  } else if (hw) {
    th = 1.0f - 2.0f * hw_rcp(hw_exp(2.0f * inner) + 1.0f);
  } else {
    const float e2x = plain_repro_exp(2.0f * inner);
    th = (e2x + -1.0f) / (e2x + 1.0f);
  }
  return 0.5f * (x * (1.0f + th));
}

enum { EXP, EXP_BR, EXP2_NEG, SIGMOID, SIGMOID_BR, SOFTPLUS, SOFTPLUS_BR, SILU, GELU, GELU_BR,
       GELU_HW, N_FORMS };

template <int F>
__device__ float plain(float x) {
  if (F == EXP || F == EXP_BR) return plain_exp(x);
  if (F == EXP2_NEG) return plain_exp2_neg(x);
  if (F == SIGMOID || F == SIGMOID_BR) return 1.0f / (1.0f + plain_exp(-x));
  if (F == SOFTPLUS || F == SOFTPLUS_BR) return plain_log(1.0f + plain_exp(x));
  if (F == SILU) return x * (1.0f / (1.0f + plain_exp(-x)));
  return plain_gelu(x, F == GELU_HW);
}

template <int F>
__device__ float kernels(float x) {
  switch (F) {
    case EXP: return expf_(x);
    case EXP_BR: return expf_br(x);
    case EXP2_NEG: return exp2_neg(x);
    case SIGMOID: return sigmoid<MATH_BF>(x);
    case SIGMOID_BR: return sigmoid<MATH_BR>(x);
    case SOFTPLUS: return softplus<MATH_BF>(x);
    case SOFTPLUS_BR: return softplus<MATH_BR>(x);
    case SILU: return silu<MATH_BF>(x);
    case GELU: return gelu<MATH_BF>(x);
    case GELU_BR: return gelu<MATH_BR>(x);
    default: return gelu<MATH_HW>(x);
  }
}

// 2^21 threads x 2^11 floats.  scatter: a wave's 64 lanes take floats 2^26
// apart, so that ordinary and special arguments meet in one wave; otherwise
// neighbours.  out: the number of floats that differ and the largest of them.
template <int F>
__global__ void check_kernel(int scatter, unsigned long long* out) {
  const uint32_t t = blockIdx.x * blockDim.x + threadIdx.x;
  for (uint32_t i = 0; i < 2048; ++i) {
    const uint32_t u = scatter ? (t & 63) << 26 | (t >> 6) << 11 | i : i << 21 | t;
    const float x = u2f(u), a = kernels<F>(x), b = plain<F>(x);
    if (f2u(a) != f2u(b) && (a == a || b == b)) {
      atomicAdd(&out[0], 1ull);
      atomicMax(&out[1], (unsigned long long)u);
    }
  }
}

template <int F>
__global__ void plain_kernel(uint32_t step, int n, float* out) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) out[i] = plain<F>(u2f((uint32_t)i * step));
}

template <int F>
hipError_t go(int form, int scatter, unsigned long long* count, uint32_t step, int n, float* y) {
  if constexpr (F < N_FORMS) {
    if (form != F) return go<F + 1>(form, scatter, count, step, n, y);
    if (count)
      hipLaunchKernelGGL(check_kernel<F>, dim3(8192), dim3(256), 0, 0, scatter, count);
    else
      hipLaunchKernelGGL(plain_kernel<F>, dim3((n + 255) / 256), dim3(256), 0, 0, step, n, y);
    return hipGetLastError();
  }
  return hipErrorInvalidValue;
}
}  // namespace

// result[0]: floats of 2^32 on which form's two functions differ, result[1]:
// the largest of them
extern "C" int math_forms_check(int form, int scatter, unsigned long long result[2]) {
  unsigned long long* d = nullptr;
  hipError_t e = hipMalloc(&d, 16);
  if (!e) e = hipMemset(d, 0, 16);
  if (!e) e = go<0>(form, scatter, d, 0, 0, nullptr);
  if (!e) e = hipMemcpy(result, d, 16, hipMemcpyDeviceToHost);
  (void)hipFree(d);
  return (int)e;
}
// out[i] = form's plain function of the float with bits i step
extern "C" int math_forms_plain(int form, uint32_t step, int n, float* out) {
  if (n < 1) return (int)hipErrorInvalidValue;
  float* d = nullptr;
  hipError_t e = hipMalloc(&d, sizeof(float) * (size_t)n);
  if (!e) e = go<0>(form, 0, nullptr, step, n, d);
  if (!e) e = hipMemcpy(out, d, sizeof(float) * (size_t)n, hipMemcpyDeviceToHost);
  (void)hipFree(d);
  return (int)e;
}
