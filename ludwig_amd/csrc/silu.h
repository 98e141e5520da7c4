// silu.h -- the activation a = bf16(z/(1 + exp(-z))), shared by the
// convolution's epilogue and the elementwise kernel, which therefore agree
// bit for bit.
//
// expf and the IEEE division cost about 45 instructions a value, most of them
// for special values: 50 of the 212 us of a 32 -> 32 layer on 8 x 64^3.
// Here -z log2(e) is formed in two parts, so that the exponential's error
// does not grow with |z|, and the hardware's reciprocal is followed by the
// division's residual step, 14 instructions; large |z|, infinities and NaN
// take expf and the division.  The BF16 result is theirs for every one of
// the 2^32 values of z (in FP32 15 differ, by at most 2 ulp).  The hardware's
// exponential and reciprocal alone, 5 instructions, would take 4 % off a layer
// on average, but are off by |z| 2^-24: 1876 of the 2^23 values in (-64, -32]
// round to the wrong BF16 value, 57 here.

#ifndef LDW_SILU_H
#define LDW_SILU_H

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace ldw {

// for |z| < 80, where no step leaves the normal range
__device__ __forceinline__ float silu_inner(float z) {
  constexpr float c = 1.44269502e+00f, cl = 1.92596303e-08f;   // log2(e) = c + cl
  // adding 1.5 2^23 rounds to an integer and leaves it in the low bits
  constexpr float magic = 12582912.0f;
  const float h = -z*c, t = h + magic;
  const float l = __builtin_fmaf(-z, cl, __builtin_fmaf(-z, c, -h));
  const float f = (h - (t - magic)) + l;
  const uint32_t e = __float_as_uint(__builtin_amdgcn_exp2f(f)) + (__float_as_uint(t) << 23);
  const float d = 1.0f + __uint_as_float(e);
  const float r = __builtin_amdgcn_rcpf(d), q = z*r;
  // (the residual this way round keeps the sign of q = -0)
  return __builtin_fmaf(-__builtin_fmaf(d, q, -z), r, q);
}

// one test for N values: a branch for each costs as much as the arithmetic
template <int N>
__device__ __forceinline__ void silu_bf16(const float (&z)[N], uint16_t (&a)[N]) {
  float m = __builtin_fabsf(z[0]);
#pragma unroll
  for (int i = 1; i < N; i++) m += __builtin_fabsf(z[i]);
  const bool inner = (m < 80.0f);
  float v[N];
  if (__builtin_expect(inner, 1)) {
#pragma unroll
    for (int i = 0; i < N; i++) v[i] = silu_inner(z[i]);
  }
  else {
#pragma unroll
    for (int i = 0; i < N; i++) v[i] = z[i]/(1.0f + expf(-z[i]));
  }
#pragma unroll
  for (int i = 0; i < N; i++) a[i] = __builtin_bit_cast(uint16_t, (__bf16) v[i]);
}

}  // namespace ldw

#endif
