// Pieces shared by the convolution kernels over few output pixels.
#pragma once

#include <algorithm>

#include "conv_common.hpp"

namespace th {

typedef _Float16 half8f __attribute__((ext_vector_type(8)));
typedef __bf16 bfloat8f __attribute__((ext_vector_type(8)));
typedef float float4f __attribute__((ext_vector_type(4)));
typedef unsigned int uint4f __attribute__((ext_vector_type(4)));
typedef unsigned int uint4f_any __attribute__((ext_vector_type(4), aligned(2)));

template <class T> __device__ inline float4f few_mfma(uint4f a, uint4f b, float4f c) {
    if constexpr (std::is_same_v<T, f16>) {
        half8f x, y;
        __builtin_memcpy(&x, &a, 16);
        __builtin_memcpy(&y, &b, 16);
        return __builtin_amdgcn_mfma_f32_16x16x32_f16(x, y, c, 0, 0, 0);
    } else {
        bfloat8f x, y;
        __builtin_memcpy(&x, &a, 16);
        __builtin_memcpy(&y, &b, 16);
        return __builtin_amdgcn_mfma_f32_16x16x32_bf16(x, y, c, 0, 0, 0);
    }
}

constexpr uint32_t kFewPitch = 20;              // floats per row of a partial 16 x 16 tile: the four row groups of a write fall on different banks

// what a block may have of LDS
constexpr size_t kFew3Lds = 160 * 1024;

}  // namespace th
