// Matrix-core operand types and the float32 operand split shared by the kernels.
#pragma once

#include "common.h"

namespace na {

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8_t;
typedef __attribute__((ext_vector_type(16))) float f32x16_t;
typedef __attribute__((ext_vector_type(8))) float f32x8_t;

// x = h[0] + h[1] + h[2], three bf16 values (rounded to nearest); exact from 2^-109 up, below
// which the last part leaves bf16's range
__device__ inline void split3(const f32x8_t& x, bf16x8_t (&h)[3]) {
  h[0] = __builtin_convertvector(x, bf16x8_t);
  const f32x8_t r = x - __builtin_convertvector(h[0], f32x8_t);
  h[1] = __builtin_convertvector(r, bf16x8_t);
  h[2] = __builtin_convertvector(r - __builtin_convertvector(h[1], f32x8_t), bf16x8_t);
}

// torch's softplus (linear above beta v = 20), branch-free; ib = 1 / beta
__device__ inline float softplus_sel(float v, float beta, float ib) {
  const float z = v * beta;
  const float r = fmaxf(v, 0.0f) + __logf(1.0f + __expf(-fabsf(z))) * ib;
  return z > 20.0f ? v : r;
}

}  // namespace na
