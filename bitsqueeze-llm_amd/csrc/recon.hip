// Low-rank reconstruction out = U diag(S) V^T, or minuend - U diag(S) V^T, on
// the f16 matrix cores with every FP32 value as two f16 pieces (h2_split.hpp)
// (reference modules/reconstruct_lowrank_cuda/src/reconstruct_lowrank_cuda.cu:
// 21-62, 120-171; the subtraction of src/bitsqz_llm.cu:1141-1163).
//
// At low ranks recon_low_rank_kernel sums in FP32 (low_rank_form, with the
// rule's reason).  Else each 128 x 128 tile of the output is one workgroup.  The
// rows of U diag(S) and of V are scaled by powers of two that bring their
// largest magnitude into [2^14, 2^15), and the tile leaves scaled back, straight
// from the accumulators: 32 lanes write 128 contiguous bytes of a row.  Two
// forms, with the same pieces summed in the same order, so with the same
// results:
//   recon_planes_kernel  where the caller has room for the pieces
//                        (FactorPlanes): factor_planes_kernel splits each
//                        factor once, from FP32 or straight from its NF4 /
//                        NF4_DQ codes, and the tiles fetch whole 16-byte units
//                        from the planes into LDS;
//   recon_kernel         without scratch: each workgroup finds the exponents
//                        of its own 256 rows, then fetches their values a
//                        slice of 32 k ahead and splits them as it stages
//                        them.
//
// Measured against the FP32 matrix cores' kernels (whose decompress side
// decoded packed factors inline), planes included: 4096 x 11008, rank 128
// 126 -> 81 us; 8192 x 4096, rank 256 167 and 171 -> 93 us; 16384 x 14336,
// rank 512 2237 and 2553 -> 890 us.  Splitting while staging in every tile
// took 96, 110 and 1182 us: twelve VALU instructions per matrix instruction.
#include "bsq_internal.hpp"
#include "h2_split.hpp"
#include "scalar_codecs.hpp"
#include "tile_map.hpp"

#include <type_traits>

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
    int m, n, k;
};

__device__ __forceinline__ int factor_exponent(uint32_t bits) {
    return bits == 0x7F800000u ? kInfRow : row_exponent(bits);
}
// scale of a row: its largest magnitude to [2^14, 2^15)
__device__ __forceinline__ float factor_scale(int e) { return pow2(14 - min(e, 127)); }

// Values k .. k + 3 of a row of K >= 4 (which may start at any multiple of four
// bytes), zero past its end, in two steps: the load, at the last four values
// where those lie past the end, and (once loads of other rows are out too) the
// turn to their places.  Guarded loads wait one for another: a ragged last
// slice by them took 4 us more at any size.
__device__ __forceinline__ void load_row4(const float *row, int k, int K, float (&v)[4]) {
    __builtin_memcpy(&v[0], __builtin_assume_aligned(row + min(k, K - 4), 4), 16);
}
__device__ __forceinline__ void turn_row4(int k, int K, float (&v)[4]) {
    const int past = max(k - (K - 4), 0);
    if (past & 1) {
        v[0] = v[1], v[1] = v[2], v[2] = v[3], v[3] = 0.0f;
    }
    if (past & 2) {
        v[0] = v[2], v[1] = v[3], v[2] = v[3] = 0.0f;
    }
    if (past >= 4) v[0] = v[1] = v[2] = v[3] = 0.0f;
}

// eight values of a row from k on, zero past the row's end
__device__ __forceinline__ void load_row8(const float *row, int k, int K, float (&v)[8]) {
    if (k + 8 <= K) {
        __builtin_memcpy(&v[0], __builtin_assume_aligned(row + k, 4), 32);
    } else {
#pragma unroll
        for (int i = 0; i < 8; ++i) v[i] = k + i < K ? row[k + i] : 0.0f;
    }
}

// The tile's way out: exponents eu, ev (LDS) of its rows and columns undo the
// scales; entries of a row or column with infinities are summed in FP32, since
// an infinity has no second piece.
template <class FU, class FV>
__device__ __forceinline__ void store_tile(const ReconArgs &g, const Sums &acc, const int *eu, const int *ev, int m0,
                                           int n0, int wave, int lane, FU &&u_at, FV &&v_at) {
    const int wm0 = (wave >> 1) * 64, wn0 = (wave & 1) * 64;
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
                const float x = __builtin_ldexpf(acc.hi[i][jj][q] + acc.lo[i][jj][q] * kLoInv,
                                                 min(er, 127) + min(ec, 127) - 28);
                if (row < g.m && col < g.n && er != kInfRow && ec != kInfRow)
                    g.out[static_cast<uint64_t>(row) * g.n + col] = g.minuend ? mv[q] - x : x;
            }
        }
    // the entries left out above, if any
    bool inf = ev[wn0 + (lane & 31)] == kInfRow || ev[wn0 + 32 + (lane & 31)] == kInfRow || eu[wm0 + lane] == kInfRow;
    if (!__any(inf)) return;
#pragma unroll 1
    for (int s = 0; s < 64; ++s) {
        const int q = s & 15, rl = wm0 + 32 * (s >> 5) + (q & 3) + 8 * (q >> 2) + g4;
        const int cl = wn0 + 32 * ((s >> 4) & 1) + (lane & 31), row = m0 + rl, col = n0 + cl;
        if (row >= g.m || col >= g.n || (eu[rl] != kInfRow && ev[cl] != kInfRow)) continue;
        float x = 0.0f;
#pragma unroll 1
        for (int t = 0; t < g.k; ++t) x = fmaf(u_at(row, t) * g.S[t], v_at(col, t), x);
        const uint64_t e = static_cast<uint64_t>(row) * g.n + col;
        g.out[e] = g.minuend ? g.minuend[e] - x : x;
    }
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
        } else if (g.k % 4 == 0) {  // uniform
            // clamped quads and selected zeros (guarded loads wait one for
            // another: 4 us more at any size)
#pragma unroll
            for (int c = 0; c < 8; c += 4) {
                const int kc = min(k + c, g.k - 4);
#pragma unroll
                for (int h = 0; h < 4; ++h) __builtin_memcpy(&v[h][c], __builtin_assume_aligned(rows[h] + kc, 4), 16);
                __builtin_memcpy(&s8[c], __builtin_assume_aligned(g.S + kc, 4), 16);
            }
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                const bool past = k + (i & 4) >= g.k;
#pragma unroll
                for (int h = 0; h < 4; ++h) v[h][i] = past ? 0.0f : v[h][i];
                s8[i] = past ? 0.0f : s8[i];
            }
        } else {
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                const int kc = min(k + i, g.k - 1);
#pragma unroll
                for (int h = 0; h < 4; ++h) v[h][i] = rows[h][kc];
                s8[i] = g.S[kc];
            }
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                const bool past = k + i >= g.k;
#pragma unroll
                for (int h = 0; h < 4; ++h) v[h][i] = past ? 0.0f : v[h][i];
                s8[i] = past ? 0.0f : s8[i];
            }
        }
    };
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

    auto at = [&](const float *f) {
        return [=](int row, int t) { return f[static_cast<uint64_t>(row) * g.k + t]; };
    };
    store_tile(g, acc, eu, ev, m0, n0, wave, lane, at(g.U), at(g.V));
}

// ---------------------------------------------------------------------------
// A factor as pieces: planes [k / 8][padded rows][8] of f16, h then l, zero
// past k and past the rows, and the exponent of each row.
struct PlaneSource {
    const float *dense;       // FP32 values, or null
    const uint8_t *codes;     // NF4 / NF4_DQ nibbles, element 2 j in the high one
    const float *scales_f32;  // NF4 block scales
    const uint8_t *scales_u8; // NF4_DQ block scale codes
    const float *dq;          // NF4_DQ global scale
    const float *S;           // values times S[k], or null
    u32x4 *h, *l;
    int *e;
    int rows, padded;
};

// scale of block b, as the decoder computes it (quantization_cuda.cu:300-305,
// 322-332)
__device__ __forceinline__ float block_scale(const PlaneSource &p, uint64_t b, float dq) {
    const float s = p.scales_u8 ? dq * e4m3_decode(p.scales_u8[b]) : p.scales_f32[b];
    return (s == 0.0f || !__builtin_isfinite(s)) ? 1.0f : s;
}

// One workgroup per 16 rows (the first `groups_u` of U, the others of V); the
// sixteen groups of sixteen lanes share a row's groups of eight k.  Exponents
// first, then the pieces, the values of up to 512 k held in registers between
// (64 rows a workgroup, each value read twice, took 22 us instead of 8 at
// 8192 x 4096, rank 256: too few loads in flight).  Quantised factors are
// decoded here, element by element as the decoder does.
constexpr int kPlaneRows = 16;
__global__ __launch_bounds__(kThreads) void factor_planes_kernel(PlaneSource u, PlaneSource v, int groups_u, int k,
                                                                 int kgroups) {
    constexpr float Lc[16] = BSQ_NF4_LEVELS;
    __shared__ float levels[16];
    __shared__ uint32_t wbits[kThreads / 64][kPlaneRows];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const bool is_u = static_cast<int>(blockIdx.x) < groups_u;  // uniform
    const PlaneSource p = is_u ? u : v;
    const int row = (static_cast<int>(blockIdx.x) - (is_u ? 0 : groups_u)) * kPlaneRows + (lane & 15);
    const int kg0 = 4 * wave + (lane >> 4);
    if (tid < 16) levels[tid] = Lc[tid];
    __syncthreads();
    const uint64_t base = static_cast<uint64_t>(min(row, p.rows - 1)) * k;
    float dq = 1.0f;
    if (p.scales_u8) {
        dq = *p.dq;
        if (dq == 0.0f || !__builtin_isfinite(dq)) dq = 1.0f;
    }
    // a group of eight in one 64-element block, its codes in one aligned word
    // (a caller's code arrays may start at any byte)
    const bool quick = k % 8 == 0 && (reinterpret_cast<uintptr_t>(p.codes) & 3u) == 0;
    auto values = [&](int kg, float (&x)[8]) {
        const int k0 = 8 * kg;
        const uint64_t e0 = base + k0;
        if (p.dense) {
            load_row8(p.dense + base, k0, k, x);
        } else if (quick && k0 < k) {
            const uint32_t w = *reinterpret_cast<const uint32_t *>(p.codes + e0 / 2);
            const float s = block_scale(p, e0 / kQuantBlock, dq);
#pragma unroll
            for (int i = 0; i < 8; ++i) x[i] = s * levels[(w >> (8 * (i / 2) + (i % 2 ? 0 : 4))) & 15u];
        } else {
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                const uint64_t e = e0 + i;
                x[i] = 0.0f;
                if (k0 + i < k) {
                    const uint32_t byte = p.codes[e >> 1];
                    x[i] = block_scale(p, e / kQuantBlock, dq) * levels[(e & 1) ? (byte & 15u) : (byte >> 4)];
                }
            }
        }
        if (p.S) {
#pragma unroll
            for (int i = 0; i < 8; ++i)
                if (k0 + i < k) x[i] *= p.S[k0 + i];
        }
    };
    constexpr int kKeep = 4, kStep = 16;  // groups of eight k held per lane, and their distance
    float x[kKeep][8];
    uint32_t bits = 0;
    auto largest = [&](const float (&y)[8]) {
#pragma unroll
        for (int i = 0; i < 8; ++i) bits = max(bits, __float_as_uint(fabsf(y[i])));
    };
#pragma unroll
    for (int n = 0; n < kKeep; ++n)
        if (kg0 + kStep * n < kgroups) values(kg0 + kStep * n, x[n]);
#pragma unroll
    for (int n = 0; n < kKeep; ++n)
        if (kg0 + kStep * n < kgroups) largest(x[n]);
    for (int kg = kg0 + kStep * kKeep; kg < kgroups; kg += kStep) {
        float y[8];
        values(kg, y);
        largest(y);
    }
    for (int off = 16; off <= 32; off <<= 1)
        bits = max(bits, static_cast<uint32_t>(__shfl_xor(static_cast<int>(bits), off)));
    if (lane < kPlaneRows) wbits[wave][lane] = bits;
    __syncthreads();
#pragma unroll
    for (int w = 0; w < kThreads / 64; ++w) bits = max(bits, wbits[w][lane & 15]);
    const int e = factor_exponent(bits);
    if (tid < kPlaneRows && row < p.rows) p.e[row] = e;
    const float sc = row < p.rows ? factor_scale(e) : 0.0f;
    auto put = [&](int kg, const float (&y)[8]) {
        u32x4 h, l;
        split8(y, [&](int) { return sc; }, h, l);
        const uint64_t unit = static_cast<uint64_t>(kg) * p.padded + row;
        p.h[unit] = h;
        p.l[unit] = l;
    };
#pragma unroll
    for (int n = 0; n < kKeep; ++n)
        if (kg0 + kStep * n < kgroups) put(kg0 + kStep * n, x[n]);
    for (int kg = kg0 + kStep * kKeep; kg < kgroups; kg += kStep) {
        float y[8];
        values(kg, y);
        put(kg, y);
    }
}

// element (row, t) of a factor, without S
__device__ float factor_value(const PlaneSource &p, int row, int t, int k) {
    constexpr float Lc[16] = BSQ_NF4_LEVELS;
    const uint64_t e = static_cast<uint64_t>(row) * k + t;
    if (p.dense) return p.dense[e];
    float dq = 1.0f;
    if (p.scales_u8) {
        dq = *p.dq;
        if (dq == 0.0f || !__builtin_isfinite(dq)) dq = 1.0f;
    }
    const uint32_t byte = p.codes[e >> 1];
    return block_scale(p, e / kQuantBlock, dq) * Lc[(e & 1) ? (byte & 15u) : (byte >> 4)];
}

struct PlaneArgs {
    PlaneSource u, v;
    int slices;  // 16-deep slices (a multiple of two)
};

typedef __attribute__((address_space(3))) void lds_void_t;
typedef __attribute__((address_space(1))) void glb_void_t;

// Slices of 16 k through a ring of four LDS stages, three in flight: wave 0
// fetches U's h units, wave 1 its l units, waves 2 and 3 V's.  One LDS object
// per stage, so that no wait is inserted for another stage's transfers.
__global__ __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(2, 2))) void recon_planes_kernel(
    ReconArgs g, PlaneArgs pl) {
    constexpr int kStage = 4 * 2 * T;  // units: planes uh, ul, vh, vl of two k groups x 128 rows
    constexpr int kDma = 4;            // transfers of a wave per slice
    __shared__ __attribute__((aligned(1024))) u32x4 st0[kStage], st1[kStage], st2[kStage], st3[kStage];
    __shared__ int eu[T], ev[T];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int wm0 = (wave >> 1) * 64, wn0 = (wave & 1) * 64;
    int tile_m, tile_n, z;
    xcd_tile(static_cast<int>(ceil_div(g.m, T)), static_cast<int>(ceil_div(g.n, T)), 1, tile_m, tile_n, z);
    const int m0 = tile_m * T, n0 = tile_n * T;
    if (tid < T) eu[tid] = pl.u.e[min(m0 + tid, g.m - 1)];
    else ev[tid - T] = pl.v.e[min(n0 + tid - T, g.n - 1)];  // both visible after the loop's barriers

    // this wave's plane, from its first row; rows past the planes repeat the
    // last 64 (their results are not stored)
    const u32x4 *src = wave == 0 ? pl.u.h : (wave == 1 ? pl.u.l : (wave == 2 ? pl.v.h : pl.v.l));
    const int rows = wave < 2 ? pl.u.padded : pl.v.padded, r0 = wave < 2 ? m0 : n0;
    const int c0 = min(r0, rows - 64) + lane, c1 = min(r0 + 64, rows - 64) + lane;
    auto issue = [&](const u32x4 *st, int j) __attribute__((always_inline)) {
        asm volatile("" ::: "memory");
#pragma unroll
        for (int kg = 0; kg < 2; ++kg) {
            const u32x4 *p = src + static_cast<uint64_t>(2 * j + kg) * rows;
            const u32x4 *dst = st + (2 * wave + kg) * T;
            __builtin_amdgcn_global_load_lds((glb_void_t *)(p + c0), (lds_void_t *)(reinterpret_cast<size_t>(dst)), 16,
                                             0, 0);
            __builtin_amdgcn_global_load_lds((glb_void_t *)(p + c1),
                                             (lds_void_t *)(reinterpret_cast<size_t>(dst + 64)), 16, 0, 0);
        }
        asm volatile("" ::: "memory");
    };
    Sums acc;
    acc.clear();
    // slice j from `cur`; slice j + 3 goes to `nxt`, read in slice j - 1.
    // Past the last slice the transfers repeat it, so the count of those in
    // flight is the same in every slice.
    auto slice = [&](const u32x4 *cur, const u32x4 *nxt, int j) __attribute__((always_inline)) {
        asm volatile("" ::: "memory");
        __builtin_amdgcn_s_waitcnt(0x070 | (2 * kDma));  // lgkmcnt(0), vmcnt(8): slice j has landed
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        issue(nxt, min(j + 3, pl.slices - 1));
        Frags f;
        const int o = (lane >> 5) * T + (lane & 31);
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            f.ah[i] = __builtin_bit_cast(f16x8, cur[o + wm0 + 32 * i]);
            f.bh[i] = __builtin_bit_cast(f16x8, cur[4 * T + o + wn0 + 32 * i]);
            f.al[i] = __builtin_bit_cast(f16x8, cur[2 * T + o + wm0 + 32 * i]);
            f.bl[i] = __builtin_bit_cast(f16x8, cur[6 * T + o + wn0 + 32 * i]);
        }
        acc.multiply(f);
    };
    issue(st0, 0);
    issue(st1, min(1, pl.slices - 1));
    issue(st2, min(2, pl.slices - 1));
    for (int j = 0; j < pl.slices; j += 4) {
        slice(st0, st3, j);
        slice(st1, st0, j + 1);
        if (j + 2 < pl.slices) {  // uniform; the slices come in pairs
            slice(st2, st1, j + 2);
            slice(st3, st2, j + 3);
        }
    }
    // no transfer into LDS outlives the workgroup
    __builtin_amdgcn_s_waitcnt(0x070);
    store_tile(
        g, acc, eu, ev, m0, n0, wave, lane, [&](int row, int t) { return factor_value(pl.u, row, t, g.k); },
        [&](int row, int t) { return factor_value(pl.v, row, t, g.k); });
}

// Low ranks on the FP32 matrix instructions: the whole of k is in LDS after one
// round trip to memory, with packed factors decoded on the way, and a 64 x 64
// tile goes out as 16-byte stores (V's rows are the instruction's rows, so a
// lane holds four consecutive columns).  Small matrices are bound by that round
// trip, large ones by the output's writes to about rank 32 and by the matrix
// instructions above.  4-byte loads and guarded tails cost more than either:
// every load and store of a tile inside the matrix is one of 16 bytes without a
// branch of its own (8192 x 8192, rank 32 86 -> 60 us, rank 48 143 -> 81).
// The order of the sums is that of gemm.hip's kernels: lane group kk takes
// k = 16 s + 4 kk + t at step t of slice s.
// QUADS: every quad of k is one load (ranks from four; of packed factors,
// multiples of four, whose quads lie in one 64-element block), else by element.
template <int KS, bool PACKED, bool SUB, bool QUADS>
__global__ __launch_bounds__(kThreads) void recon_low_rank_kernel(ReconArgs g, PlaneSource u, PlaneSource v) {
    constexpr int TS = 64, G = 4 * KS;  // quads of k per row
    constexpr int KP = 16 * KS + 4, Q = TS * G / kThreads, F = TS / 32;
    constexpr float Lc[16] = BSQ_NF4_LEVELS;
    __shared__ __attribute__((aligned(16))) float us[TS][KP], vs[TS][KP];
    __shared__ float levels[16];
    int tile_m, tile_n, z;
    xcd_tile(static_cast<int>(ceil_div(g.m, TS)), static_cast<int>(ceil_div(g.n, TS)), 1, tile_m, tile_n, z);
    const int m0 = tile_m * TS, n0 = tile_n * TS, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, K = g.k;
    if constexpr (PACKED) {
        if (tid < 16) levels[tid] = Lc[tid];
        __syncthreads();
    }
    // the quads of a factor's rows from row r0 on; rows past the factor repeat
    // its last one.  Quads that reach past k are loaded where they end at it
    // and turned to their places by stage().
    auto load = [&](const PlaneSource &p, int r0, float (&x)[Q][4]) __attribute__((always_inline)) {
        const bool packed = PACKED && !p.dense;
        float dq = 1.0f;
        if (packed && p.scales_u8) {
            dq = *p.dq;
            if (dq == 0.0f || !__builtin_isfinite(dq)) dq = 1.0f;
        }
        const bool words = (reinterpret_cast<uintptr_t>(p.codes) & 1u) == 0;
#pragma unroll
        for (int q = 0; q < Q; ++q) {
            const int lin = tid + kThreads * q, k0 = 4 * (lin % G);
            const uint64_t base = static_cast<uint64_t>(min(r0 + lin / G, p.rows - 1)) * K;
            if (!packed && QUADS) {
                load_row4(p.dense + base, k0, K, x[q]);
            } else if (QUADS) {
                const uint64_t e = base + min(k0, K - 4);
                const uint8_t *c = p.codes + e / 2;
                const uint32_t w = words ? *reinterpret_cast<const uint16_t *>(c) : c[0] | (c[1] << 8);
                const float s = block_scale(p, e / kQuantBlock, dq);
#pragma unroll
                for (int i = 0; i < 4; ++i) x[q][i] = s * levels[(w >> (8 * (i / 2) + (i % 2 ? 0 : 4))) & 15u];
            } else {
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const uint64_t e = base + min(k0 + i, K - 1);
                    if (!packed) {
                        x[q][i] = p.dense[e];
                    } else {
                        const uint32_t byte = p.codes[e >> 1];
                        x[q][i] = block_scale(p, e / kQuantBlock, dq) * levels[(e & 1) ? (byte & 15u) : (byte >> 4)];
                    }
                }
            }
        }
    };
    auto stage = [&](float (&x)[Q][4], float (*dst)[KP]) __attribute__((always_inline)) {
        if (QUADS && K % 4 != 0) {  // uniform
#pragma unroll
            for (int q = 0; q < Q; ++q) turn_row4(4 * ((tid + kThreads * q) % G), K, x[q]);
        }
#pragma unroll
        for (int q = 0; q < Q; ++q) {
            const int lin = tid + kThreads * q, k0 = 4 * (lin % G);
            f32x4 y;
#pragma unroll
            for (int i = 0; i < 4; ++i) y[i] = k0 + i < K ? x[q][i] : 0.0f;
            *reinterpret_cast<f32x4 *>(&dst[lin / G][k0]) = y;
        }
    };
    {
        float xu[Q][4], xv[Q][4], xs[Q][4];
        load(u, m0, xu);
        load(v, n0, xv);
#pragma unroll
        for (int q = 0; q < Q; ++q) {
            const int k0 = 4 * ((tid + kThreads * q) % G);
            if (QUADS) {
                load_row4(g.S, k0, K, xs[q]);
            } else {
#pragma unroll
                for (int i = 0; i < 4; ++i) xs[q][i] = g.S[min(k0 + i, K - 1)];
            }
        }
#pragma unroll
        for (int q = 0; q < Q; ++q)
#pragma unroll
            for (int i = 0; i < 4; ++i) xu[q][i] *= xs[q][i];
        stage(xu, us);
        stage(xv, vs);
    }
    __syncthreads();
    const int row0 = (wave >> 1) * 32 + (lane & 15), col0 = (wave & 1) * 32, kk = lane >> 4;
    const bool inside = m0 + TS <= g.m && n0 + TS <= g.n;  // uniform
    auto at = [&](int i, int j) {  // column block i, row block j
        return static_cast<uint64_t>(m0 + row0 + 16 * j) * g.n + (n0 + col0 + 16 * i + 4 * kk);
    };
    // (rows of out and minuend may start at any multiple of four bytes)
    f32x4 acc[F][F], mv[F][F];
#pragma unroll
    for (int j = 0; j < F; ++j)
#pragma unroll
        for (int i = 0; i < F; ++i) {
            acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
            if (SUB && inside) __builtin_memcpy(&mv[i][j], __builtin_assume_aligned(g.minuend + at(i, j), 4), 16);
        }
#pragma unroll
    for (int s = 0; s < KS; ++s) {
        f32x4 a[F], b[F];
#pragma unroll
        for (int i = 0; i < F; ++i) {
            a[i] = *reinterpret_cast<const f32x4 *>(&vs[col0 + 16 * i + (lane & 15)][16 * s + 4 * kk]);
            b[i] = *reinterpret_cast<const f32x4 *>(&us[row0 + 16 * i][16 * s + 4 * kk]);
        }
#pragma unroll
        for (int t = 0; t < 4; ++t)
#pragma unroll
            for (int i = 0; i < F; ++i)
#pragma unroll
                for (int j = 0; j < F; ++j)
                    acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[i][t], b[j][t], acc[i][j], 0, 0, 0);
    }
    if (inside) {
#pragma unroll
        for (int j = 0; j < F; ++j)
#pragma unroll
            for (int i = 0; i < F; ++i) {
                const f32x4 x = SUB ? mv[i][j] - acc[i][j] : acc[i][j];
                __builtin_memcpy(__builtin_assume_aligned(g.out + at(i, j), 4), &x, 16);
            }
        return;
    }
#pragma unroll
    for (int j = 0; j < F; ++j)
#pragma unroll
        for (int i = 0; i < F; ++i) {
            const int row = m0 + row0 + 16 * j, col = n0 + col0 + 16 * i + 4 * kk;
            if (row >= g.m) continue;
#pragma unroll
            for (int t = 0; t < 4; ++t)
                if (col + t < g.n) g.out[at(i, j) + t] = SUB ? g.minuend[at(i, j) + t] - acc[i][j][t] : acc[i][j][t];
        }
}

template <bool PACKED, bool SUB>
void low_rank(const ReconArgs &g, const PlaneSource &u, const PlaneSource &v, hipStream_t stream) {
    const dim3 grid(static_cast<unsigned>(ceil_div(g.m, 64) * ceil_div(g.n, 64)));
    auto go = [&](auto kern) { kern<<<grid, kThreads, 0, stream>>>(g, u, v); };
    auto depth = [&](auto quads) {
        constexpr bool Q = decltype(quads)::value;
        if (g.k <= 16) go(recon_low_rank_kernel<1, PACKED, SUB, Q>);
        else if constexpr (PACKED || Q) {
            if (g.k <= 32) go(recon_low_rank_kernel<2, PACKED, SUB, Q>);
            else if (g.k <= 48) go(recon_low_rank_kernel<3, PACKED, SUB, Q>);
            else if (g.k <= 64) go(recon_low_rank_kernel<4, PACKED, SUB, Q>);
            else if (g.k <= 96) go(recon_low_rank_kernel<6, PACKED, SUB, Q>);
            else go(recon_low_rank_kernel<8, PACKED, SUB, Q>);
        }
    };
    if (PACKED ? g.k % 4 == 0 : g.k >= 4) depth(std::true_type{});
    else depth(std::false_type{});
    BSQ_HIP(hipGetLastError());
}

void launch_low_rank(const ReconArgs &g, const PlaneSource &u, const PlaneSource &v, hipStream_t stream) {
    const bool dense = u.dense && v.dense;
    if (g.minuend) {
        if (dense) low_rank<false, true>(g, u, v, stream);
        else low_rank<true, true>(g, u, v, stream);
    } else {
        if (dense) low_rank<false, false>(g, u, v, stream);
        else low_rank<true, false>(g, u, v, stream);
    }
}

}  // namespace

namespace {
// Which form a shape takes, with scratch or without, so that both give the same
// bits.  FP32 sums to rank 64 at any size (8192 x 8192, rank 48 81 us against
// 102 from two slices of pieces, rank 64 96 and 98; 512 x 1024, rank 64 4.4 and
// 11.2), and to rank 128 while the 128 x 128 tiles of the other form would leave
// CUs idle (2048 x 2048, 256 tiles, rank 128 14.7 and 16.5 us, rank 80 12.8 and
// 16.2; 2048 x 4096, rank 80 21.8 and 19.5).
bool low_rank_form(int m, int n, int k) {
    return k <= 64 || (k <= 128 && ceil_div(m, T) * ceil_div(n, T) <= static_cast<uint64_t>(cu_count()));
}
// Whether packed factors are decoded ahead of the low-rank kernel (two launches,
// 5 us) and not in each tile, which costs 0.012 us per rank and tile a CU:
// 4096 x 4096, rank 64 39 us against 46, rank 8 27 against 25.
bool decodes_first(int m, int n, int k) {
    return ceil_div(m, 64) * ceil_div(n, 64) * k > 400ull * cu_count();
}
uint64_t dense_bytes(int rows, int k) { return ceil_div(static_cast<uint64_t>(rows) * k, 4) * 16; }
int padded_rows(int rows) { return static_cast<int>(ceil_div(rows, 64) * 64); }
int plane_groups(int k) { return static_cast<int>(ceil_div(k, BK) * KG); }
}  // namespace

uint64_t factor_plane_bytes(int m, int n, int k) {
    if (low_rank_form(m, n, k)) return decodes_first(m, n, k) ? dense_bytes(m, k) + dense_bytes(n, k) : 0;
    return 2ull * 16 * plane_groups(k) * (static_cast<uint64_t>(padded_rows(m)) + padded_rows(n)) +
           sizeof(int) * (static_cast<uint64_t>(m) + n);
}

void launch_reconstruct(const float *U, const float *S, const float *V, int m, int n, int k, const float *minuend,
                        float *out, hipStream_t stream) {
    BSQ_REQUIRE(m > 0 && n > 0 && k > 0 && U && S && V && out, "reconstruct: bad arguments");
    const ReconArgs g{U, S, V, minuend, out, m, n, k};
    if (low_rank_form(m, n, k)) {
        launch_low_rank(g, PlaneSource{U, nullptr, nullptr, nullptr, nullptr, nullptr, nullptr, nullptr, nullptr, m, 0},
                        PlaneSource{V, nullptr, nullptr, nullptr, nullptr, nullptr, nullptr, nullptr, nullptr, n, 0},
                        stream);
        return;
    }
    recon_kernel<<<static_cast<unsigned>(ceil_div(m, T) * ceil_div(n, T)), kThreads, 0, stream>>>(g);
    BSQ_HIP(hipGetLastError());
}

void launch_reconstruct_planes(const FactorSource &U, const float *S, const FactorSource &V, int m, int n, int k,
                               const float *minuend, float *out, void *planes, hipStream_t stream) {
    BSQ_REQUIRE(m > 0 && n > 0 && k > 0 && S && out && (planes || factor_plane_bytes(m, n, k) == 0),
                "reconstruct: bad arguments");
    for (const FactorSource *f : {&U, &V})
        BSQ_REQUIRE(f->dense || (f->codes && (f->scales_f32 || (f->scales_u8 && f->dq))), "reconstruct: missing factor");
    if (low_rank_form(m, n, k)) {
        auto source = [&](const FactorSource &f, int rows, uint64_t at) {
            const float *dense = f.dense;
            if (!dense && decodes_first(m, n, k)) {
                auto *to = reinterpret_cast<float *>(static_cast<uint8_t *>(planes) + at);
                launch_quant_decode(static_cast<uint64_t>(rows) * k, f.scales_u8 ? kMethodNF4DQ : kMethodNF4,
                                    f.scales_f32, f.scales_u8, f.dq, f.codes, to, stream);
                dense = to;
            }
            return PlaneSource{dense, f.codes, f.scales_f32, f.scales_u8, f.dq, nullptr, nullptr, nullptr, nullptr,
                               rows, 0};
        };
        const PlaneSource u = source(U, m, 0), v = source(V, n, dense_bytes(m, k));
        launch_low_rank(ReconArgs{nullptr, S, nullptr, minuend, out, m, n, k}, u, v, stream);
        return;
    }
    const int kgroups = plane_groups(k), up = padded_rows(m), vp = padded_rows(n);
    auto *uh = static_cast<u32x4 *>(planes);
    u32x4 *ul = uh + static_cast<uint64_t>(kgroups) * up, *vh = ul + static_cast<uint64_t>(kgroups) * up,
          *vl = vh + static_cast<uint64_t>(kgroups) * vp;
    int *eu = reinterpret_cast<int *>(vl + static_cast<uint64_t>(kgroups) * vp), *ev = eu + m;
    const PlaneSource pu{U.dense, U.codes, U.scales_f32, U.scales_u8, U.dq, S, uh, ul, eu, m, up};
    const PlaneSource pv{V.dense, V.codes, V.scales_f32, V.scales_u8, V.dq, nullptr, vh, vl, ev, n, vp};
    factor_planes_kernel<<<static_cast<unsigned>((up + vp) / kPlaneRows), kThreads, 0, stream>>>(
        pu, pv, up / kPlaneRows, k, kgroups);
    BSQ_HIP(hipGetLastError());
    const ReconArgs g{nullptr, S, nullptr, minuend, out, m, n, k};
    const PlaneArgs pl{pu, pv, kgroups / 2};
    recon_planes_kernel<<<static_cast<unsigned>(ceil_div(m, T) * ceil_div(n, T)), kThreads, 0, stream>>>(g, pl);
    BSQ_HIP(hipGetLastError());
}

}  // namespace bsq
