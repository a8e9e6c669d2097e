/*
 * F32 operands of BF16 matrix instructions (softmax weights, states, decays): two BF16 numbers each, the value rounded and what the
 * rounding left (16 bits together), two values at a time so that each conversion instruction makes two of them.
 */
#ifndef GD_OPS_SHARED_HIP_WEIGHT_PAIRS_H
#define GD_OPS_SHARED_HIP_WEIGHT_PAIRS_H
#include "hip_device.h"

typedef float gd_float2v __attribute__((ext_vector_type(2)));

/* elements at, at + 1 of two vectors */
template <typename V>
__device__ __forceinline__ void gd_weight_pair(float a, float b, V &rounded, V &rest, int at)
{
    union { gd_bf16x2 h; uint32_t u; } r, s;
    r.h = __builtin_convertvector((gd_float2v){a, b}, gd_bf16x2);
    s.h = __builtin_convertvector((gd_float2v){a - __uint_as_float(r.u << 16), b - __uint_as_float(r.u & 0xffff0000u)}, gd_bf16x2);
    rounded[at] = r.h[0];
    rounded[at + 1] = r.h[1];
    rest[at] = s.h[0];
    rest[at + 1] = s.h[1];
}

#endif
