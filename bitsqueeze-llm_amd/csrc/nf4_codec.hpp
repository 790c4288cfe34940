// NF4 / NF4_DQ element encoding shared by the quantiser (quant.hip) and the
// fused encode + error top-k pass (topk.hip): the reference's nearest-level
// rule (quantization_cuda.cu:43-58) with its tie behaviour, and the NF4_DQ
// global scale (quantization_cuda.cu:222-249).
#pragma once

#include "bsq_internal.hpp"

namespace bsq {
namespace {

__device__ __forceinline__ float sanitize(float x) { return __builtin_isfinite(x) ? x : 0.0f; }

// The reference's linear scan: first index minimising |fl(v - L[i])|
// (quantization_cuda.cu:43-58).  Used only where |v| >= 2 or v is not finite.
__device__ __noinline__ uint32_t nf4_code_scan(float v) {
    constexpr float L[16] = BSQ_NF4_LEVELS;
    if (!__builtin_isfinite(v)) v = 0.0f;
    uint32_t best = 0;
    float best_err = fabsf(v - L[0]);
#pragma unroll
    for (int i = 1; i < 16; ++i) {
        const float err = fabsf(v - L[i]);
        if (err < best_err) {
            best_err = err;
            best = i;
        }
    }
    return best;
}

// The same scan over the levels held in `L` (LDS), inline and not unrolled:
// a call to the out-of-line scan from a kernel that holds many values in
// registers makes the compiler park them in callee-saved registers around
// the call, which spreads them over far more registers than they need.
__device__ __forceinline__ uint32_t nf4_code_scan_inline(const float *L, float v) {
    if (!__builtin_isfinite(v)) v = 0.0f;
    uint32_t best = 0;
    float best_err = fabsf(v - L[0]);
#pragma unroll 1
    for (int i = 1; i < 16; ++i) {
        const float err = fabsf(v - L[i]);
        if (err < best_err) {
            best_err = err;
            best = static_cast<uint32_t>(i);
        }
    }
    return best;
}

// Nearest NF4 code with the reference's tie rule: for |v| < 2 the scan's
// answer is the number of exact decision thresholds at or below v, found
// here with one table lookup and one comparison.  [-1, 2) is cut into 48
// bins of width 1/16; bin b holds code_lo = #{T_i <= -1 + b/16} and the
// threshold lying inside the bin, if any (no bin holds two: the closest
// thresholds are 0.081 apart).  Every threshold is at least 1.6e-3 from a bin
// edge, while the bin index floor((v + 1) * 16), computed in FP32 with one
// rounding or two, is off by one only for v within 1.2e-7 of an edge, where
// the count is the same on both sides; v in (-2, -1] takes bin 0, and the
// largest v below 2 rounds up to bin 48, which holds code 15 as the bins
// before it do.  |v| >= 2 and non-finite v take the scan.  Both forms of the
// bin are checked exhaustively against the scan over all 2^32 floats by the
// GPU test suite.  So few bins span one and a half
// rounds of the LDS banks: 384 bins of 1/128 took 93 us against 85 in the
// fused encode and top-k pass of 4096 x 11008 (with its other changes).
constexpr int kNf4PerUnit = 16, kNf4Bins = 3 * kNf4PerUnit + 1;
struct Nf4Table {
    uint2 ent[kNf4Bins];  // (bits of the threshold inside bin b, code_lo): one 8-byte read
};

// the table's entries, computed by the compiler
struct Nf4TableValues {
    float thr[kNf4Bins];
    uint32_t lo[kNf4Bins];
    constexpr Nf4TableValues() : thr(), lo() {
        constexpr float T[15] = BSQ_NF4_THRESHOLDS;
        for (int b = 0; b < kNf4Bins; ++b) {
            const float e0 = -1.0f + static_cast<float>(b) / kNf4PerUnit, e1 = -1.0f + static_cast<float>(b + 1) / kNf4PerUnit;
            thr[b] = __builtin_inff();
            for (int i = 0; i < 15; ++i) {
                lo[b] += T[i] <= e0 ? 1u : 0u;
                if (T[i] > e0 && T[i] < e1) thr[b] = T[i];
            }
        }
    }
};
__device__ const Nf4TableValues kNf4TableValues{};

__device__ __forceinline__ void nf4_table_build(Nf4Table &t) {
    for (int b = threadIdx.x; b < kNf4Bins; b += blockDim.x)
        t.ent[b] = uint2{__float_as_uint(kNf4TableValues.thr[b]), kNf4TableValues.lo[b]};
}

// the table path alone: |v| < 2
__device__ __forceinline__ uint32_t nf4_code_small(const Nf4Table &t, float v) {
    const int b = min(max(static_cast<int>((v + 1.0f) * static_cast<float>(kNf4PerUnit)), 0), kNf4Bins - 1);
    const uint2 e = t.ent[b];
    return e.y + ((v >= __uint_as_float(e.x)) ? 1u : 0u);
}

// bin of x inv, |x inv| < 2, given inv_bins = kNf4PerUnit inv: one FMA and one
// conversion (which takes negative values and NaN to 0).  The sum rounds to
// 3 kNf4PerUnit at most, the table's last entry.
__device__ __forceinline__ uint32_t nf4_bin(float x, float inv_bins) {
    const float t = __builtin_fmaf(x, inv_bins, static_cast<float>(kNf4PerUnit));
    uint32_t b;
    asm("v_cvt_u32_f32 %0, %1" : "=v"(b) : "v"(t));
    return b;
}

// code of x inv, |x inv| < 2 (NaN: 0)
__device__ __forceinline__ uint32_t nf4_code_binned(const Nf4Table &t, float x, float inv, float inv_bins) {
    const uint2 e = t.ent[nf4_bin(x, inv_bins)];
    return e.y + ((x * inv >= __uint_as_float(e.x)) ? 1u : 0u);
}

// Largest magnitude of v[0 .. N), and whether any of them is NaN; infinities
// give infinity.  (N even: two values an instruction.)
template <int N>
__device__ __forceinline__ float magnitude_max(const float (&v)[N], bool &nan) {
    float m = 0.0f;
    nan = false;
#pragma unroll
    for (int i = 0; i < N; i += 2) {
        asm("v_max3_f32 %0, |%1|, |%2|, %0" : "+v"(m) : "v"(v[i]), "v"(v[i + 1]));
        nan = nan || __builtin_isunordered(v[i], v[i + 1]);
    }
    return m;
}

__device__ __forceinline__ uint32_t nf4_code(const Nf4Table &t, float v) {
    if (fabsf(v) < 2.0f) return nf4_code_small(t, v);
    return nf4_code_scan(v);
}

__device__ __forceinline__ float dq_raw_from_gmax(uint32_t gbits) {
    // store_dq_scale_kernel (quantization_cuda.cu:222-233)
    const float g = __uint_as_float(gbits);
    if (g == 0.0f || !__builtin_isfinite(g)) return 1.0f;
    return g / kE4M3Max;
}

__device__ __forceinline__ float dq_effective(float dq) {
    // nf4_dq_compress_kernel / nf4_dq_decompress_kernel (quantization_cuda.cu:246-249, 324-327)
    return (dq == 0.0f || !__builtin_isfinite(dq)) ? 1.0f : dq;
}

}  // namespace
}  // namespace bsq
