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

// two values x, scaled by f, to their pieces, packed.  Three mixed-precision
// FMAs a value write the pieces into their halves (h = f16(f x), f x - h
// exactly, l = f16 of 2^11 times that); left to the compiler it is five
// instructions, with the products and the packing of their own.
__device__ __forceinline__ void split2(float x0, float x1, float f0, float f1, uint32_t &h, uint32_t &l) {
    uint32_t hp, lp;
    float r0, r1;
    asm("v_fma_mixlo_f16 %0, %1, %2, 0" : "=v"(hp) : "v"(x0), "v"(f0));
    asm("v_fma_mixhi_f16 %0, %1, %2, 0" : "+v"(hp) : "v"(x1), "v"(f1));
    asm("v_fma_mix_f32 %0, %1, %2, -%3 op_sel_hi:[0,0,1]" : "=v"(r0) : "v"(x0), "v"(f0), "v"(hp));
    asm("v_fma_mix_f32 %0, %1, %2, -%3 op_sel:[0,0,1] op_sel_hi:[0,0,1]" : "=v"(r1) : "v"(x1), "v"(f1), "v"(hp));
    asm("v_fma_mixlo_f16 %0, %1, %2, 0" : "=v"(lp) : "v"(r0), "s"(kLo));
    asm("v_fma_mixhi_f16 %0, %1, %2, 0" : "+v"(lp) : "v"(r1), "s"(kLo));
    h = hp;
    l = lp;
}

// eight values x, scaled by f, to their pieces
template <class F>
__device__ __forceinline__ void split8(const float (&x)[8], F &&f, u32x4 &h, u32x4 &l) {
#pragma unroll
    for (int p = 0; p < 4; ++p) {
        uint32_t hp, lp;
        split2(x[2 * p], x[2 * p + 1], f(2 * p), f(2 * p + 1), hp, lp);
        h[p] = hp;
        l[p] = lp;
    }
}

// The range finder's small operand B (an orthonormal basis or the sketch):
// scaled by 2^kScaleB, and in products with A^T its row k also by
// 2^(E[k] - emax) (E, emax: the row exponents of A and their maximum).
constexpr int kScaleB = 11;
__device__ __forceinline__ float b_scale(const int *__restrict__ E, int emax, int k) {
    return E ? pow2(max(E[k] - emax, -138) + kScaleB) : static_cast<float>(1 << kScaleB);
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
