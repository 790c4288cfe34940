// Low-rank reconstruction out = U diag(S) V^T, or minuend - U diag(S) V^T, on
// the f16 matrix cores with every FP32 value as two f16 pieces (h2_split.hpp)
// (reference modules/reconstruct_lowrank_cuda/src/reconstruct_lowrank_cuda.cu:
// 21-62, 120-171; the subtraction of src/bitsqz_llm.cu:1141-1163).
//
// Each 128 x 128 tile of the output is one workgroup.  The rows of U diag(S)
// and of V are scaled by powers of two that bring their largest magnitude into
// [2^14, 2^15); their values are fetched a slice of 32 k ahead, split and
// staged into LDS planes, and the tile leaves scaled back, straight from the
// accumulators: 32 lanes write 128 contiguous bytes of a row.  The exponents
// of the rows come from factor_exponent_kernel where the caller has room for
// them, else each workgroup finds those of its own 256 rows first; the values
// are the same, so the results are too.
//
// Measured against the FP32 matrix cores' kernels (which also decoded packed
// factors inline on the decompress side): 4096 x 11008, rank 128 126 -> 96 us;
// 8192 x 4096, rank 256 167 and 171 -> 110 us; 16384 x 14336, rank 512 2237
// and 2553 -> 1234 us.
#include "bsq_internal.hpp"
#include "h2_split.hpp"
#include "tile_map.hpp"

namespace bsq {
namespace {

constexpr int kThreads = 256;
constexpr int T = 128, BK = 32, KG = BK / 8;
constexpr int kPitch = 130;      // 16-byte units per k group of a plane (128 rows, padded)
constexpr int kInfRow = 128;     // "exponent" of a row that holds infinities and no NaN

struct ReconArgs {
    const float *U, *S, *V;
    const float *minuend;  // or null
    float *out;
    const int *eu, *ev;    // row exponents, or null
    int m, n, k;
};

__device__ __forceinline__ int factor_exponent(uint32_t bits) {
    return bits == 0x7F800000u ? kInfRow : row_exponent(bits);
}
// scale of a row: its largest magnitude to [2^14, 2^15)
__device__ __forceinline__ float factor_scale(int e) { return pow2(14 - min(e, 127)); }

// eight values of a row from k on (rows may start at any multiple of four
// bytes), zero past the row's end
__device__ __forceinline__ void load_row8(const float *row, int k, int K, float (&v)[8]) {
    if (k + 8 <= K) {
        __builtin_memcpy(&v[0], __builtin_assume_aligned(row + k, 4), 32);
    } else {
#pragma unroll
        for (int i = 0; i < 8; ++i) v[i] = k + i < K ? row[k + i] : 0.0f;
    }
}

// exponents of the rows of U diag(S) (e[0 .. m)) and of V (e[m .. m + n)):
// one wave per row
__global__ __launch_bounds__(kThreads) void factor_exponent_kernel(const float *__restrict__ U,
                                                                   const float *__restrict__ S,
                                                                   const float *__restrict__ V, int m, int n, int k,
                                                                   int *__restrict__ e) {
    const int r = blockIdx.x * (kThreads / 64) + (threadIdx.x >> 6), lane = threadIdx.x & 63;
    if (r >= m + n) return;  // whole waves
    const float *row = r < m ? U + static_cast<uint64_t>(r) * k : V + static_cast<uint64_t>(r - m) * k;
    uint32_t bits = 0;
#pragma unroll 4
    for (int c = lane; c < k; c += 64) {
        const float x = r < m ? row[c] * S[c] : row[c];
        bits = max(bits, __float_as_uint(fabsf(x)));
    }
    for (int off = 32; off >= 1; off >>= 1)
        bits = max(bits, static_cast<uint32_t>(__shfl_xor(static_cast<int>(bits), off)));
    if (lane == 0) e[r] = factor_exponent(bits);
}

// (two waves per SIMD asked for: 128 accumulators and two slices' fragments)
__global__ __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(2, 2))) void recon_kernel(ReconArgs g) {
    __shared__ u32x4 a0[2 * KG * kPitch], a1[2 * KG * kPitch];  // U diag(S): h plane, l plane
    __shared__ u32x4 b0[2 * KG * kPitch], b1[2 * KG * kPitch];  // V
    __shared__ int eu[T], ev[T];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int wm0 = (wave >> 1) * 64, wn0 = (wave & 1) * 64;
    int tile_m, tile_n, z;
    xcd_tile(static_cast<int>(ceil_div(g.m, T)), static_cast<int>(ceil_div(g.n, T)), 1, tile_m, tile_n, z);
    const int m0 = tile_m * T, n0 = tile_n * T, nk = static_cast<int>(ceil_div(g.k, BK));

    // a lane stages eight consecutive k (group kg of a slice) of rows r and
    // r + 64 of each operand; rows past the factors repeat the last one
    const int r = tid >> 2, kg = tid & 3;
    const float *rows[4] = {g.U + static_cast<uint64_t>(min(m0 + r, g.m - 1)) * g.k,
                            g.U + static_cast<uint64_t>(min(m0 + 64 + r, g.m - 1)) * g.k,
                            g.V + static_cast<uint64_t>(min(n0 + r, g.n - 1)) * g.k,
                            g.V + static_cast<uint64_t>(min(n0 + 64 + r, g.n - 1)) * g.k};
    float v[4][8], s8[8];
    auto load = [&](int j) __attribute__((always_inline)) {
        const int k = j * BK + 8 * kg;
        if ((j + 1) * BK <= g.k) {  // uniform: every slice but a ragged last one
#pragma unroll
            for (int h = 0; h < 4; ++h) __builtin_memcpy(&v[h][0], __builtin_assume_aligned(rows[h] + k, 4), 32);
            __builtin_memcpy(&s8[0], __builtin_assume_aligned(g.S + k, 4), 32);
        } else {
#pragma unroll
            for (int h = 0; h < 4; ++h) load_row8(rows[h], k, g.k, v[h]);
            load_row8(g.S, k, g.k, s8);
        }
    };
    if (g.eu) {  // uniform
        if (tid < T) eu[tid] = g.eu[min(m0 + tid, g.m - 1)];
        else ev[tid - T] = g.ev[min(n0 + tid - T, g.n - 1)];
    } else {
        uint32_t bits[4] = {0, 0, 0, 0};
        for (int j = 0; j < nk; ++j) {
            load(j);
#pragma unroll
            for (int h = 0; h < 4; ++h)
#pragma unroll
                for (int i = 0; i < 8; ++i)
                    bits[h] = max(bits[h], __float_as_uint(fabsf(h < 2 ? v[h][i] * s8[i] : v[h][i])));
        }
#pragma unroll
        for (int h = 0; h < 4; ++h) {
            for (int off = 1; off <= 2; off <<= 1)
                bits[h] = max(bits[h], static_cast<uint32_t>(__shfl_xor(static_cast<int>(bits[h]), off)));
            if (kg == 0) (h < 2 ? eu : ev)[64 * (h & 1) + r] = factor_exponent(bits[h]);
        }
    }
    load(0);
    __syncthreads();
    float sc[4];
#pragma unroll
    for (int h = 0; h < 4; ++h) sc[h] = factor_scale((h < 2 ? eu : ev)[64 * (h & 1) + r]);

    auto stage = [&](u32x4 *as, u32x4 *bs) __attribute__((always_inline)) {
#pragma unroll
        for (int h = 0; h < 4; ++h) {
            float x[8];
#pragma unroll
            for (int i = 0; i < 8; ++i) x[i] = h < 2 ? v[h][i] * s8[i] : v[h][i];
            u32x4 hp, lp;
            split8(x, [&](int) { return sc[h]; }, hp, lp);
            u32x4 *dst = (h < 2 ? as : bs) + kg * kPitch + 64 * (h & 1) + r;
            dst[0] = hp;
            dst[KG * kPitch] = lp;
        }
    };
    Sums acc;
    acc.clear();
    auto fetch = [&](Frags &f, const u32x4 *as, const u32x4 *bs, int s) __attribute__((always_inline)) {
        const int o = (2 * s + (lane >> 5)) * kPitch + (lane & 31);
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            f.ah[i] = __builtin_bit_cast(f16x8, as[o + wm0 + 32 * i]);
            f.bh[i] = __builtin_bit_cast(f16x8, bs[o + wn0 + 32 * i]);
            f.al[i] = __builtin_bit_cast(f16x8, as[KG * kPitch + o + wm0 + 32 * i]);
            f.bl[i] = __builtin_bit_cast(f16x8, bs[KG * kPitch + o + wn0 + 32 * i]);
        }
    };
    // slice j is in the current stage once every wave has passed the barrier;
    // the next one goes to the other stage, read in slice j - 1, while this
    // one is multiplied
    auto slice = [&](u32x4 *ac, u32x4 *bc, u32x4 *an, u32x4 *bn, int j) __attribute__((always_inline)) {
        asm volatile("" ::: "memory");
        __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0): the fetched values stay in flight
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        if (j + 1 < nk) {  // uniform
            stage(an, bn);
            load(min(j + 2, nk - 1));
        }
        Frags f;
        fetch(f, ac, bc, 0);
        acc.multiply(f);
        fetch(f, ac, bc, 1);
        acc.multiply(f);
    };
    stage(a0, b0);
    load(min(1, nk - 1));
    for (int j = 0; j < nk; j += 2) {
        slice(a0, b0, a1, b1, j);
        if (j + 1 < nk) slice(a1, b1, a0, b0, j + 1);
    }

    const int g4 = 4 * (lane >> 5);
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int jj = 0; jj < 2; ++jj) {
            const int cl = wn0 + 32 * jj + (lane & 31), col = n0 + cl;
            const int ec = ev[cl];
            float mv[16];
            if (g.minuend) {  // uniform
#pragma unroll
                for (int q = 0; q < 16; ++q) {
                    const int row = min(m0 + wm0 + 32 * i + (q & 3) + 8 * (q >> 2) + g4, g.m - 1);
                    mv[q] = g.minuend[static_cast<uint64_t>(row) * g.n + min(col, g.n - 1)];
                }
            }
#pragma unroll
            for (int q = 0; q < 16; ++q) {
                const int rl = wm0 + 32 * i + (q & 3) + 8 * (q >> 2) + g4, row = m0 + rl;
                const int er = eu[rl];
                float x = __builtin_ldexpf(acc.hi[i][jj][q] + acc.lo[i][jj][q] * kLoInv,
                                           min(er, 127) + min(ec, 127) - 28);
                if (er == kInfRow || ec == kInfRow) {
                    // an infinity has no second piece: these entries in FP32
                    const float *u = g.U + static_cast<uint64_t>(min(row, g.m - 1)) * g.k;
                    const float *w = g.V + static_cast<uint64_t>(min(col, g.n - 1)) * g.k;
                    x = 0.0f;
#pragma unroll 1
                    for (int t = 0; t < g.k; ++t) x = fmaf(u[t] * g.S[t], w[t], x);
                }
                if (row < g.m && col < g.n)
                    g.out[static_cast<uint64_t>(row) * g.n + col] = g.minuend ? mv[q] - x : x;
            }
        }
}

// Ranks below 32: FP32 sums over k.  There the two pieces' own rounding (7e-8
// of the result) is no smaller than an FP32 chain's, and a full slice would be
// mostly padding.  64 x 64 tiles, 4 x 4 outputs a lane, the factors in LDS.
__global__ __launch_bounds__(kThreads) void recon_low_rank_kernel(ReconArgs g) {
    constexpr int TS = 64;
    __shared__ float us[BK][TS + 4], vs[BK][TS + 4];
    int tile_m, tile_n, z;
    xcd_tile(static_cast<int>(ceil_div(g.m, TS)), static_cast<int>(ceil_div(g.n, TS)), 1, tile_m, tile_n, z);
    const int m0 = tile_m * TS, n0 = tile_n * TS, tid = threadIdx.x;
    for (int e = tid; e < TS * g.k; e += kThreads) {
        const int r = e / g.k, t = e - r * g.k;
        us[t][r] = g.U[static_cast<uint64_t>(min(m0 + r, g.m - 1)) * g.k + t] * g.S[t];
        vs[t][r] = g.V[static_cast<uint64_t>(min(n0 + r, g.n - 1)) * g.k + t];
    }
    __syncthreads();
    const int r0 = 4 * (tid >> 4), c0 = 4 * (tid & 15);
    float acc[4][4] = {};
    for (int t = 0; t < g.k; ++t) {
        const float4 u = *reinterpret_cast<const float4 *>(&us[t][r0]), w = *reinterpret_cast<const float4 *>(&vs[t][c0]);
        const float uu[4] = {u.x, u.y, u.z, u.w}, ww[4] = {w.x, w.y, w.z, w.w};
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int j = 0; j < 4; ++j) acc[i][j] = fmaf(uu[i], ww[j], acc[i][j]);
    }
    const bool vec = g.n % 4 == 0 && (reinterpret_cast<uintptr_t>(g.out) & 15u) == 0 &&
                     (reinterpret_cast<uintptr_t>(g.minuend) & 15u) == 0;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int row = m0 + r0 + i, col = n0 + c0;
        if (row >= g.m || col >= g.n) continue;
        const uint64_t e = static_cast<uint64_t>(row) * g.n + col;
        if (vec) {  // whole quads: n % 4 == 0
            float4 x{acc[i][0], acc[i][1], acc[i][2], acc[i][3]};
            if (g.minuend) {
                const float4 mv = *reinterpret_cast<const float4 *>(g.minuend + e);
                x = float4{mv.x - x.x, mv.y - x.y, mv.z - x.z, mv.w - x.w};
            }
            *reinterpret_cast<float4 *>(g.out + e) = x;
        } else {
#pragma unroll
            for (int j = 0; j < 4; ++j)
                if (col + j < g.n) g.out[e + j] = g.minuend ? g.minuend[e + j] - acc[i][j] : acc[i][j];
        }
    }
}

}  // namespace

void launch_reconstruct(const float *U, const float *S, const float *V, int m, int n, int k, const float *minuend,
                        float *out, int *exponents, hipStream_t stream) {
    BSQ_REQUIRE(m > 0 && n > 0 && k > 0 && U && S && V && out, "reconstruct: bad arguments");
    ReconArgs g{U, S, V, minuend, out, exponents, exponents ? exponents + m : nullptr, m, n, k};
    if (k < BK) {
        recon_low_rank_kernel<<<static_cast<unsigned>(ceil_div(m, 64) * ceil_div(n, 64)), kThreads, 0, stream>>>(g);
        BSQ_HIP(hipGetLastError());
        return;
    }
    if (exponents) {
        factor_exponent_kernel<<<static_cast<unsigned>(ceil_div(static_cast<uint64_t>(m) + n, kThreads / 64)), kThreads,
                                 0, stream>>>(U, S, V, m, n, k, exponents);
        BSQ_HIP(hipGetLastError());
    }
    recon_kernel<<<static_cast<unsigned>(ceil_div(m, T) * ceil_div(n, T)), kThreads, 0, stream>>>(g);
    BSQ_HIP(hipGetLastError());
}

}  // namespace bsq
