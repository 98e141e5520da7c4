// silu.h -- the activation a = bf16(z/(1 + exp(-z))), shared by the
// convolution's epilogue and the elementwise kernel, which therefore agree
// bit for bit.
//
// The exponential and the reciprocal are the hardware's (1 ulp each, the
// exponent's rounding adds |z| 2^-24): the result is rounded to 8 bits
// anyway.  Over 2^24 normal z of sigma 0.5 to 30 the 2-norm error against 64
// bits is 1.66e-3 of the values, the same to 7 digits as with expf and an
// IEEE division, which cost about 45 instructions a value where this costs
// 7: they were 50 of the 212 us of a 32 -> 32 layer on 8 x 64^3.  Below
// z = -88 the result is -0 instead of some -1e-37.

#ifndef LDW_SILU_H
#define LDW_SILU_H

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace ldw {

__device__ __forceinline__ uint16_t silu_bf16(float z) {
  return __builtin_bit_cast(uint16_t, (__bf16) (z*__builtin_amdgcn_rcpf(1.0f + __expf(-z))));
}

}  // namespace ldw

#endif
