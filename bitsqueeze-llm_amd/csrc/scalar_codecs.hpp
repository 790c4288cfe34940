// Scalar FP8 E4M3 codec shared by the NF4_DQ block scales (quant.hip) and the
// legacy FP8 / MXFP8 / NVFP4 formats (legacy.hip).  The reference writes the
// same encoder in quantization_cuda.cu:64-109 and, identically, in
// legacy_modules/quantization/src/impl/fp8_impl.cpp:51-82,
// mxfp8_impl.cpp:56-87 and nvfp4_impl.cpp:62-93 (saturation at 448, frexp
// split, round-to-nearest-even mantissa, subnormal mantissa clamped at 7);
// the decoder has no NaN code (0x7F decodes to 480).
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

#include "bsq_internal.hpp"

namespace bsq {

// The value whose conversion to E4M3 (round to nearest even) is the code of
// quantization_cuda.cu:64-109: +-448 at most (NaN and infinities included, NaN
// positive), and below the normal range (2^-6) at most the largest subnormal
// 7 / 512, as the code's mantissa is clamped at 7 there.
__device__ __forceinline__ float e4m3_operand(float value) {
    const float w = fmaxf(fminf(value, kE4M3Max), -kE4M3Max);  // fminf takes NaN to 448
    constexpr float kMinNormal = 0.015625f, kMaxSub = 0.013671875f;
    return fabsf(w) < kMinNormal ? __builtin_amdgcn_fmed3f(w, -kMaxSub, kMaxSub) : w;
}

// FP8 E4M3 encode exactly as quantization_cuda.cu:64-109 writes it, on the
// converter (v_cvt_pk_fp8_f32); 25 instructions a value with frexp and rint,
// six here.
__device__ __forceinline__ uint32_t e4m3_encode(float value) {
    const float w = e4m3_operand(value);
    return static_cast<uint32_t>(__builtin_amdgcn_cvt_pk_fp8_f32(w, w, 0, false)) & 0xFFu;
}

// four codes, the first in the low byte
__device__ __forceinline__ uint32_t e4m3_encode4(float a, float b, float c, float d) {
    const int lo = __builtin_amdgcn_cvt_pk_fp8_f32(e4m3_operand(a), e4m3_operand(b), 0, false);
    return static_cast<uint32_t>(__builtin_amdgcn_cvt_pk_fp8_f32(e4m3_operand(c), e4m3_operand(d), lo, true));
}

// FP8 E4M3 decode (quantization_cuda.cu:111-128); 0x7F decodes to 480.  The
// code's exponent and mantissa read as FP32's are 2^-120 of the value, with
// subnormals for subnormals.
__device__ __forceinline__ float e4m3_decode(uint32_t v) {
    return __uint_as_float(static_cast<uint32_t>(static_cast<int32_t>(v << 24) >> 4) & 0x87F00000u) * 0x1.0p120f;
}

}  // namespace bsq
