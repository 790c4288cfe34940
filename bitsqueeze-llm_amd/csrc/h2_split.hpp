// FP32 values as two f16 pieces for the f16 matrix cores, shared by the
// kernels that multiply them (gemm_h2.hip, recon.hip).
//
// A value x, scaled by an exact power of two s, is h + l 2^-11 with
// h = f16(s x) and l = f16(2^11 (s x - h)): 22 bits and a sign, the rest at
// most half a unit in the last place of FP32.  A product of two such values
// is summed as
//     hi += h_a h_b          lo += h_a l_b + l_a h_b
// in FP32 accumulators of their own (v_mfma_f32_32x32x16_f16) and is
// hi + 2^-11 lo; the dropped l_a l_b is 2^-24 of the product or less, with
// either sign.  Keeping the two sums apart keeps l a normal f16 down to 2^-29
// of the scaled maximum and adds the small terms without rounding them into
// the large sum.  Against 64-bit sums the error is 0.35 to 0.9 times that of
// a v_mfma_f32_16x16x4f32 chain of the same length (K = 32 .. 11008; normal,
// lognormal, one-signed and decaying operands, and a column 10^6 times the
// others that the other operand does not touch).
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

namespace bsq {
namespace {

typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

constexpr float kLo = 2048.0f, kLoInv = 1.0f / 2048.0f;

// exponent of the largest magnitude of a row, from its bits (which order as
// the magnitudes do, NaN above infinity): in [-112, 127]; a zero row, or one
// below 2^-112, takes -112, a row with infinities or NaN 127
__device__ __forceinline__ int row_exponent(uint32_t bits) {
    return min(max(static_cast<int>(bits >> 23) - 127, -112), 127);
}

// 2^e, e in [-149, 127]
__device__ __forceinline__ float pow2(int e) { return __builtin_ldexpf(1.0f, e); }

// eight scaled values to their pieces
__device__ __forceinline__ void split8(const float (&y)[8], u32x4 &h, u32x4 &l) {
#pragma unroll
    for (int p = 0; p < 4; ++p) {
        const f16x2 hp{static_cast<_Float16>(y[2 * p]), static_cast<_Float16>(y[2 * p + 1])};
        const f16x2 lp{static_cast<_Float16>((y[2 * p] - static_cast<float>(hp.x)) * kLo),
                       static_cast<_Float16>((y[2 * p + 1] - static_cast<float>(hp.y)) * kLo)};
        h[p] = __builtin_bit_cast(uint32_t, hp);
        l[p] = __builtin_bit_cast(uint32_t, lp);
    }
}

// The matrix instructions of one 16-deep step of a wave's 64 x 64 block, from
// LDS planes [k group][row] of 16-byte units (eight consecutive k of a row):
// lane l takes row l % 32 of a 32-row block and k group l / 32, and holds of
// a 32 x 32 result column l % 32 and rows (q & 3) + 8 (q >> 2) + 4 (l / 32).
struct Frags {
    f16x8 ah[2], al[2], bh[2], bl[2];
};

struct Sums {
    f32x16 hi[2][2], lo[2][2];
    __device__ __forceinline__ void clear() {
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int j = 0; j < 2; ++j) hi[i][j] = lo[i][j] = f32x16{};
    }
    __device__ __forceinline__ void multiply(const Frags &f) {
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int j = 0; j < 2; ++j)
                hi[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(f.ah[i], f.bh[j], hi[i][j], 0, 0, 0);
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int j = 0; j < 2; ++j)
                lo[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(f.ah[i], f.bl[j], lo[i][j], 0, 0, 0);
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int j = 0; j < 2; ++j)
                lo[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(f.al[i], f.bh[j], lo[i][j], 0, 0, 0);
    }
};

}  // namespace
}  // namespace bsq
