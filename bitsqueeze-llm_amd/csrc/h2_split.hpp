// FP32 values as two f16 pieces for the f16 matrix cores, shared by the
// kernels that multiply them (gemm_h2.hip, recon.hip).
//
// A value x, scaled by an exact power of two s, is h + l 2^-11 with
// h = f16(s x) and l = f16(2^11 (s x - h)): 22 bits and a sign, one bit fewer
// than FP32 has.  Three quarters of the significands come out exact, the others
// one unit in the last place of FP32 off.  A product of two such values is
// summed as
//     hi += h_a h_b          lo += h_a l_b + l_a h_b
// in FP32 accumulators of their own (v_mfma_f32_32x32x16_f16) and is
// hi + 2^-11 lo; the dropped l_a l_b reaches 2^-22 of the product and is 2^-25
// of it in the mean, with either sign.  Keeping the two sums apart keeps l a
// normal f16 down to 2^-29 of the scaled maximum and adds the small terms
// without rounding them into the large sum.  Values below 2^-28 of their row's
// maximum (in A^T B, times the row's share of the matrix's) lose further bits;
// what they add to a sum lies below its FP32 rounding unless the other operand
// is zero on all that is larger.
//
// The sums decide the error, not the pieces: for 1000 products of activations
// with outlier columns the pieces alone are 7e-9 of the result off, rounding
// the result to FP32 2e-8, the matrix instructions' sums 1e-7 and a chain of
// FP32 additions 4e-7.  Held by tests against 64-bit results: 0.35 to 0.56 of
// an FP32 chain's error (K = 136 .. 1030; normal, lognormal, one-signed and
// decaying operands and outlier columns, single products and whole
// factorisations).  Against the library's FP32 kernels, factorisations of eleven
// shapes from 128 x 128 to 16384 x 14336 at ranks 8 to 512 with three inputs
// each: U S V^T 0.39 to 1.0 of their error in every one; U and V 0.15 to 1.0,
// but up to 1.6 at 1000 x 1003 rank 8 with outlier columns left in (2e-7 and
// 1e-7); S within two units of the last place, where the FP32 kernels' was
// within one.
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
