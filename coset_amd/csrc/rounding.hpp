// rounding.hpp -- fp32 helpers shared by the kernels: conversion to bf16 and
// compensated sums.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace coset {

// fp32 -> bf16 round-to-nearest-even (NaN kept quiet).
__device__ __forceinline__ uint16_t f32_to_bf16(float f)
{
    uint32_t u = __float_as_uint(f);
    if ((u & 0x7fffffffu) > 0x7f800000u) return (uint16_t)((u >> 16) | 0x40u);
    u += 0x7fffu + ((u >> 16) & 1u);
    return (uint16_t)(u >> 16);
}

__device__ __forceinline__ uint32_t pack_bf16(float lo, float hi)
{
    return (uint32_t)f32_to_bf16(lo) | ((uint32_t)f32_to_bf16(hi) << 16);
}

// acc + low <- acc + low + w with the rounding error of acc + w kept in low
// (Knuth's two-sum)
__device__ __forceinline__ void two_sum(float& acc, float& low, float w)
{
    const float t = __fadd_rn(acc, w), b = __fsub_rn(t, acc);
    low = __fadd_rn(low, __fadd_rn(__fsub_rn(acc, __fsub_rn(t, b)), __fsub_rn(w, b)));
    acc = t;
}

// The sum: acc where it is not finite (low is then NaN)
__device__ __forceinline__ float two_sum_value(float acc, float low)
{
    return low - low == 0.f ? __fadd_rn(acc, low) : acc;
}

}  // namespace coset
