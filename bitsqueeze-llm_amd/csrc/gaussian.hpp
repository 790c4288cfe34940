// N(0, 1) draws: Philox4x32-10 counter-based generator + Box-Muller.
#pragma once
#include <hip/hip_runtime.h>

#include <cstdint>

namespace bsq {
namespace {

// Philox4x32-10 (Salmon, Moraes, Dror, Shaw, "Parallel random numbers: as
// easy as 1, 2, 3", SC'11): counter = element group index, key = seed.
__device__ __forceinline__ uint4 philox4x32_10(uint4 c, uint2 k) {
    constexpr uint32_t M0 = 0xD2511F53u, M1 = 0xCD9E8D57u, W0 = 0x9E3779B9u, W1 = 0xBB67AE85u;
#pragma unroll
    for (int r = 0; r < 10; ++r) {
        const uint32_t hi0 = __umulhi(M0, c.x), lo0 = M0 * c.x;
        const uint32_t hi1 = __umulhi(M1, c.z), lo1 = M1 * c.z;
        c = make_uint4(hi1 ^ c.y ^ k.x, lo1, hi0 ^ c.w ^ k.y, lo0);
        k.x += W0;
        k.y += W1;
    }
    return c;
}

// N(0, 1) draws 4 g .. 4 g + 3: Box-Muller on (r.x, r.y) and (r.z, r.w), u1 in (0, 1]
__device__ __forceinline__ void gaussian_group(uint64_t g, uint64_t seed, float (&v)[4]) {
    const uint4 r = philox4x32_10(make_uint4(static_cast<uint32_t>(g), static_cast<uint32_t>(g >> 32), 0u, 0u),
                                  make_uint2(static_cast<uint32_t>(seed), static_cast<uint32_t>(seed >> 32)));
    constexpr float kInv32 = 2.3283064365386963e-10f;
    constexpr float kTwoPi = 6.283185307179586f;
    const float u1 = (static_cast<float>(r.x) + 1.0f) * kInv32, u2 = static_cast<float>(r.y) * kInv32;
    const float u3 = (static_cast<float>(r.z) + 1.0f) * kInv32, u4 = static_cast<float>(r.w) * kInv32;
    const float ra = sqrtf(-2.0f * logf(fminf(u1, 1.0f))), rb = sqrtf(-2.0f * logf(fminf(u3, 1.0f)));
    float s1, c1, s2, c2;
    sincosf(kTwoPi * u2, &s1, &c1);
    sincosf(kTwoPi * u4, &s2, &c2);
    v[0] = ra * c1;
    v[1] = ra * s1;
    v[2] = rb * c2;
    v[3] = rb * s2;
}

// draws 0 .. n - 1 into out, by lane `at` of `lanes`
__device__ __forceinline__ void gaussian_fill(float *__restrict__ out, uint64_t n, uint64_t seed, uint64_t at,
                                              uint64_t lanes) {
    for (uint64_t g = at; 4 * g < n; g += lanes) {
        float v[4];
        gaussian_group(g, seed, v);
#pragma unroll
        for (int i = 0; i < 4; ++i)
            if (4 * g + i < n) out[4 * g + i] = v[i];
    }
}

}  // namespace
}  // namespace bsq
