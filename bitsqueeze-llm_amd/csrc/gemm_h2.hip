// Products with the big activation matrix on the f16 matrix cores, each FP32
// operand value carried as two f16 pieces (v_mfma_f32_32x32x16_f16).
//
//   C[M x N] = op(A)[M x K] * B[K x N]     (row-major, FP32 in and out)
//     op(A) = A    (TA = false, A is M x K)      the range finder's A_w B and
//     op(A) = A^T  (TA = true,  A is K x M)      A_w^T B, A read in place
//
// The split and its error: h2_split.hpp.
// Three f16 products run at up to 5 times the FP32 matrix rate (2.5 / 3
// against 0.157 PFLOP/s).  Measured, against the FP32 kernels with their
// reductions: 4096 x 11008 with q = 128 101 -> 47 us (A^T B) and 98 -> 47 us
// (A B); 16384 x 14336 with q = 512 1986 -> 838 and 1590 -> 825 us, 0.86
// PFLOP/s of f16 products (a large library bf16 product reaches 1.2 on this
// card).  There the clock falls to 1.9 GHz (2.3 to 2.5 in the memory-bound and
// one-workgroup kernels beside them) and the matrix cores are busy in 0.43 to
// 0.5 of the cycles.
//
// Scales.  Row i of A is scaled so that its largest magnitude falls in
// [2^14, 2^15) (row_scale_kernel, once per matrix).  With TA = false that is
// a scale per row of C, undone with the partial sums' reduction.  With TA =
// true the rows run along K: B's row i takes the inverse power times
// 2^(E_max) (E_max the exponent of the largest entry of A), so the product
// needs one common factor.  B (an orthonormal basis or the sketch, entries
// below 32) is scaled by 2^11 and split ahead into planes [k / 8][column][8]
// whose 16-byte units go to LDS as they lie: by the orthonormalisation that
// makes it (chol_solve_kernel, k <= 256) or by split_b_kernel.  A is split as
// it is staged.  K is padded to pairs of slices: B's planes hold zeros there
// and A's loads repeat values of the same row or column.  (The reduction added
// the last K % 64 products in FP32, one by one: 1000 x 1003, rank 8, a whole
// round trip 408 us, padded 318.)  A small matrix's factorisation is bound by
// its launches: planes written by the orthonormalisation, the sketch drawn in
// row_scale_kernel's launch and the scales' maximum taken in split_b_kernel's
// replace 2 niter + 2 of them (4096 x 4096, rank 8, niter 2, a round trip 505
// -> 476 us, rank 256 1946 -> 1933).  All scalings are exact.  Rows holding
// infinities or NaN give NaN results, as sums over them do.
#include "bsq_internal.hpp"
#include "gaussian.hpp"
#include "h2_split.hpp"
#include "tile_map.hpp"

#include <algorithm>

namespace bsq {
namespace {

typedef __attribute__((address_space(3))) void lds_void_t;
typedef __attribute__((address_space(1))) void glb_void_t;

constexpr int kThreads = 256;
constexpr int T = 128;        // output tile
constexpr int BK = 32;        // K slice
constexpr int KG = BK / 8;    // groups of eight k per slice

__device__ __forceinline__ void dma16(const u32x4 *g, const u32x4 *l) {
    __builtin_amdgcn_global_load_lds((glb_void_t *)(g), (lds_void_t *)(reinterpret_cast<size_t>(l)), 16, 0, 0);
}

// all LDS operations of this wave and all but its PENDING newest vector
// memory operations are done, then the workgroup barrier
template <int PENDING>
__device__ __forceinline__ void stage_barrier() {
    static_assert(PENDING >= 0 && PENDING < 64, "vmcnt has six bits");
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt(0x070 | (PENDING & 15) | ((PENDING >> 4) << 14));
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
}

// Row exponents and scales of a row-major matrix: rs[i] = 2^(14 - E_i) scales
// row i into f16's range, ri[i] = 2^(E_i - 14 - kScaleB) undoes it together
// with B's scale.  One workgroup per row: the matrix is read once, at the
// rate of a copy's reads.  Workgroups past the last row draw the sketch (fill
// values into R), which needs nothing of A.
__global__ __launch_bounds__(kThreads) void row_scale_kernel(const float *__restrict__ A, int rows, int cols,
                                                             int *__restrict__ E, float *__restrict__ rs,
                                                             float *__restrict__ ri, float *__restrict__ R,
                                                             uint64_t fill, uint64_t seed) {
    __shared__ uint32_t wmax[kThreads / 64];
    const int r = blockIdx.x, tid = threadIdx.x;
    if (r >= rows) {  // uniform
        gaussian_fill(R, fill, seed, static_cast<uint64_t>(r - rows) * kThreads + tid,
                      static_cast<uint64_t>(gridDim.x - rows) * kThreads);
        return;
    }
    const float *row = A + static_cast<uint64_t>(r) * cols;
    uint32_t m = 0;  // bit patterns of magnitudes order as the magnitudes do, NaN above infinity
    const int head = min(cols, static_cast<int>((16 - (reinterpret_cast<uintptr_t>(row) & 15u)) & 15u) / 4);
    if (tid < head) m = __float_as_uint(fabsf(row[tid]));
    const float4 *q = reinterpret_cast<const float4 *>(row + head);
    const int n4 = (cols - head) / 4;
#pragma unroll 4
    for (int i = tid; i < n4; i += kThreads) {
        const float4 v = q[i];
        m = max(max(m, __float_as_uint(fabsf(v.x))), __float_as_uint(fabsf(v.y)));
        m = max(max(m, __float_as_uint(fabsf(v.z))), __float_as_uint(fabsf(v.w)));
    }
    const int t0 = head + 4 * n4;
    if (tid < cols - t0) m = max(m, __float_as_uint(fabsf(row[t0 + tid])));
    for (int off = 32; off >= 1; off >>= 1) m = max(m, static_cast<uint32_t>(__shfl_xor(static_cast<int>(m), off)));
    if ((tid & 63) == 0) wmax[tid >> 6] = m;
    __syncthreads();
    if (tid == 0) {
        m = max(max(wmax[0], wmax[1]), max(wmax[2], wmax[3]));
        const int e = row_exponent(m);
        E[r] = e;
        rs[r] = pow2(14 - e);
        ri[r] = pow2(e - 14 - kScaleB);
    }
}

// B (K x N, row-major) into its two planes, [k / 8][np][8] f16 each, kgroups
// groups of k, zero beyond row K and column N: entry (k, n) times b_scale, at
// place (k + rot) % 8 of its group if that is the partial one.
// One lane per column and group of eight k.  With rows > 0 the maximum of E's
// first `rows` entries is not yet known: the workgroups that need it find it
// (E, at most a few tens of KB, comes from L2), and the first leaves it and
// pow2(max - 14 - kScaleB) in emax and common.
__global__ __launch_bounds__(kThreads) void split_b_kernel(const float *__restrict__ B, int K, int N, int np, int kgroups,
                                                           int rot,
                                                           const int *__restrict__ E, int rows, bool scaled,
                                                           int *__restrict__ emax, float *__restrict__ common,
                                                           u32x4 *__restrict__ hi, u32x4 *__restrict__ lo) {
    __shared__ int wmax[kThreads / 64];
    int em = 0;
    if (rows > 0 && (scaled || blockIdx.x == 0)) {  // uniform
        em = -112;
#pragma unroll 8
        for (int i = threadIdx.x; i < rows; i += kThreads) em = max(em, E[i]);
        for (int off = 32; off >= 1; off >>= 1) em = max(em, __shfl_xor(em, off));
        if ((threadIdx.x & 63) == 0) wmax[threadIdx.x >> 6] = em;
        __syncthreads();
        em = max(max(wmax[0], wmax[1]), max(wmax[2], wmax[3]));
        if (blockIdx.x == 0 && threadIdx.x == 0) {
            *emax = em;
            *common = pow2(em - 14 - kScaleB);
        }
    } else if (scaled) {
        em = *emax;
    }
    if (kgroups == 0) return;  // the maximum alone (a caller's sketch): no planes, np is 0
    const int t = blockIdx.x * kThreads + threadIdx.x;
    const int kg = t / np, n = t - kg * np;
    if (kg >= kgroups) return;
    float y[8];
    const int turn = kg == K / 8 ? rot : 0;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        const int k = 8 * kg + ((i - turn) & 7);
        y[i] = n < N && k < K ? B[static_cast<uint64_t>(k) * N + n] : 0.0f;
    }
    u32x4 h, l;
    split8(y, [&](int i) { return b_scale(scaled ? E : nullptr, em, min(8 * kg + i, K - 1)); }, h, l);
    hi[t] = h;
    lo[t] = l;
}

struct H2Args {
    const float *A;
    const u32x4 *bh, *bl;  // B's planes
    const float *rs;       // scales of A's rows
    float *ws;             // partial tiles [tile row][tile column][part][tile]
    int M, N, K, lda;
    int np;                // columns of the planes (a multiple of 64)
    int tiles_n;           // output tiles per row of tiles
    int pairs;             // pairs of K slices per tile
    int units;             // tile rows x pairs
    int ranges;            // contiguous shares of the units
    int maxparts;          // workspace slots per tile
};

// range that holds unit u
__host__ __device__ __forceinline__ int h2_owner(int64_t u, int64_t units, int ranges) {
    return static_cast<int>(((u + 1) * ranges - 1) / units);
}

// Stream-K: the K slices of all tile rows, in pairs, are cut into equal
// contiguous ranges; the tiles_n workgroups of a range run the same slices of
// A against their own columns of B, side by side on one XCD, so they share A
// in its L2 (16384 x 14336 with q = 512: 1.4 GB come from HBM for A B, of which
// A is 0.94, and 4.5 GB for A^T B).  Each workgroup writes its partial sum of
// every tile it touches and h2_reduce_kernel adds a tile's parts in order.
//
// 128 x 128 tiles, four waves of 64 x 64 in 32 x 32 blocks with both sums in
// accumulator registers (128 of 256 a lane), so two workgroups share a CU and
// one's staging and barriers run under the other's matrix instructions.
// 128 x 256 and 256 x 128 tiles (one workgroup a CU, three quarters of the
// operand bytes per product) measured the same within 3 %, as one 128 x 128
// workgroup a CU does.  Slices of 32 k: B's pieces go global -> LDS directly one
// slice ahead; A's values are fetched into registers two slices ahead (row-major: a
// lane takes eight consecutive k of two rows; A^T: eight k-rows of two
// columns, so the transposition is only a choice of registers), then split and
// written to LDS in the same [k group][row] units of 16 bytes that the
// fragments are read in.
template <bool TA>
__global__ __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(2, 2))) void gemm_h2_kernel(H2Args g) {
    constexpr int kPitchA = T + 2;  // 16-byte units per k group of a staged A plane: +2 spreads the writes' banks
    __shared__ u32x4 a0[2 * KG * kPitchA], a1[2 * KG * kPitchA];  // h plane, l plane
    __shared__ __attribute__((aligned(1024))) u32x4 b0[2 * KG * T], b1[2 * KG * T];
    // vector loads of one A slice's values, at least: 16 bytes are the widest
    // (32 bytes a lane of each of two rows), and A^T's are one row apart, a
    // runtime stride.  Their addresses differ by lane, so none is a scalar load.
    constexpr int kLoadsA = TA ? 16 : 4;

    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int wm0 = (wave >> 1) * 64, wn0 = (wave & 1) * 64;
    const int G = static_cast<int>(gridDim.x), bid = static_cast<int>(blockIdx.x);
    const int xcd = bid % kXcds, loc = bid / kXcds;
    const int L = xcd * (G / kXcds) + min(xcd, G % kXcds) + loc;
    const int range = L / g.tiles_n, tn = L - range * g.tiles_n;
    const int p0 = static_cast<int>(static_cast<int64_t>(range) * g.units / g.ranges);
    const int n = static_cast<int>(static_cast<int64_t>(range + 1) * g.units / g.ranges) - p0;  // slice pairs

    // a position in the slices of the range (tile row, slice), `left` slices
    // before its last
    struct Cursor {
        int tm, ks, left;
        __device__ __forceinline__ void next(int nk) {
            // by selects: branches here would split the accumulators' live ranges
            const int step = left > 0 ? 1 : 0;
            left -= step;
            const int w = ks + step == nk ? 1 : 0;
            ks = w ? 0 : ks + step;
            tm += w;
        }
    };
    const int nk = 2 * g.pairs, tile0 = p0 / g.pairs;
    Cursor ca{tile0, 2 * (p0 - tile0 * g.pairs), 2 * n - 1};  // next A slice to fetch
    Cursor cb = ca;                                           // next B slice to fetch

    float va[2][8];  // A values in flight
    float vs[TA ? 8 : 2];
    auto load_a = [&]() __attribute__((always_inline)) {
        const int m0 = ca.tm * T, k0 = ca.ks * BK;
        asm volatile("" ::: "memory");  // stays behind the DMA before it
        if constexpr (!TA) {
#pragma unroll
            for (int h = 0; h < 2; ++h) vs[h] = g.rs[min(m0 + 64 * h + (tid >> 2), g.M - 1)];
            asm volatile("" ::: "memory");  // the scales first: the wait lets values alone stay in flight
            const int k = min(k0 + 8 * (tid & 3), g.K - 8);
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const int r = min(m0 + 64 * h + (tid >> 2), g.M - 1);
                // past K: the row's last eight values, which meet a partial
                // group of B turned to fit them (H2Planes), or zeros
                // rows may start at any multiple of four bytes
                __builtin_memcpy(&va[h][0], __builtin_assume_aligned(g.A + static_cast<uint64_t>(r) * g.lda + k, 4), 32);
            }
        } else {
            // k-rows are the wave's own: scalar bases, one 32-bit offset a column
            uint32_t c[2];
#pragma unroll
            for (int h = 0; h < 2; ++h) c[h] = 4u * static_cast<uint32_t>(min(m0 + 64 * h + lane, g.M - 1));
#pragma unroll
            for (int i = 0; i < 8; ++i) vs[i] = g.rs[min(k0 + 8 * wave + i, g.K - 1)];
            const int k = k0 + 8 * __builtin_amdgcn_readfirstlane(wave);
            const char *p = reinterpret_cast<const char *>(g.A) + 4u * static_cast<uint64_t>(min(k, g.K - 1)) * g.lda;
#pragma unroll
            for (int i = 0; i < 8; ++i) {
#pragma unroll
                for (int h = 0; h < 2; ++h) va[h][i] = *reinterpret_cast<const float *>(p + c[h]);
                // past K: the last row again, against zeros of B
                p += k + i + 1 < g.K ? 4u * static_cast<uint64_t>(g.lda) : 0u;
            }
        }
        ca.next(nk);
    };
    auto stage_a = [&](u32x4 *as) __attribute__((always_inline)) {
        const int row = TA ? lane : tid >> 2, kg = TA ? wave : tid & 3;
        // the values are first touched here: their scaling, moved up past the
        // barrier, would wait for them a slice early
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
            for (int i = 0; i < 8; ++i) asm volatile("" : "+v"(va[h][i]));
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            u32x4 hp, lp;
            split8(va[h], [&](int i) { return TA ? vs[i] : vs[h]; }, hp, lp);
            as[kg * kPitchA + 64 * h + row] = hp;
            as[(KG + kg) * kPitchA + 64 * h + row] = lp;
        }
    };
    auto dma_b = [&](const u32x4 *bs) __attribute__((always_inline)) {  // wave w: k group w of both planes
        asm volatile("" ::: "memory");
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const int nc = min(tn * T + 64 * h, g.np - 64);  // beyond the planes: results not stored
            const uint64_t src = static_cast<uint64_t>(cb.ks * KG + wave) * g.np + nc + lane;
            dma16(g.bh + src, bs + wave * T + 64 * h);
            dma16(g.bl + src, bs + (KG + wave) * T + 64 * h);
        }
        asm volatile("" ::: "memory");
        cb.next(nk);
    };

    Sums acc;
    auto fetch = [&](Frags &f, const u32x4 *as, const u32x4 *bs, int s) __attribute__((always_inline)) {
        const int kg = 2 * s + (lane >> 5), r = lane & 31;
#pragma unroll
        for (int i = 0; i < 2; ++i) f.ah[i] = __builtin_bit_cast(f16x8, as[kg * kPitchA + wm0 + 32 * i + r]);
#pragma unroll
        for (int j = 0; j < 2; ++j) f.bh[j] = __builtin_bit_cast(f16x8, bs[kg * T + wn0 + 32 * j + r]);
#pragma unroll
        for (int j = 0; j < 2; ++j) f.bl[j] = __builtin_bit_cast(f16x8, bs[(KG + kg) * T + wn0 + 32 * j + r]);
#pragma unroll
        for (int i = 0; i < 2; ++i) f.al[i] = __builtin_bit_cast(f16x8, as[(KG + kg) * kPitchA + wm0 + 32 * i + r]);
    };

    // the partial tile of tile row t goes out, in 16-byte units in accumulator
    // order: [wave][i][j][q / 4][lane]
    auto flush = [&](int t) __attribute__((always_inline)) {
        const int first = h2_owner(static_cast<int64_t>(t) * g.pairs, g.units, g.ranges);
        uint32_t unit = static_cast<uint32_t>(wave) * (T * T / 16) + static_cast<uint32_t>(lane);
        asm volatile("" : "+v"(unit));  // the addresses are formed here, not held through the loop
        f32x4 *W = reinterpret_cast<f32x4 *>(g.ws) +
                   ((static_cast<uint64_t>(t) * g.tiles_n + tn) * g.maxparts + (range - first)) * (T * T / 4) + unit;
#pragma unroll
        for (int i = 0; i < 2; ++i)
            for (int jj = 0; jj < 2; ++jj) {
                if (tn * T + wn0 + 32 * jj >= g.N) continue;  // uniform: columns past C's
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    f32x4 v;
#pragma unroll
                    for (int e = 0; e < 4; ++e)
                        v[e] = acc.hi[i][jj][4 * q + e] + acc.lo[i][jj][4 * q + e] * kLoInv;
                    W[((2 * i + jj) * 4 + q) * 64] = v;
                }
            }
    };

    // a slice: its A and B are in the current stage once every wave has
    // passed the barrier, which also frees the other stage (read one slice
    // ago); the next slice's A is in registers or in flight behind this
    // slice's B (and is staged before B's next transfers are issued: the
    // compiler's wait for it takes everything in flight).  Nothing in a
    // slice is conditional, which would split the accumulators' live ranges:
    // past the range's end the fetches repeat its last slice.
    auto slice = [&](u32x4 *ac, u32x4 *bc, u32x4 *an, u32x4 *bn) __attribute__((always_inline)) {
        stage_barrier<kLoadsA>();
        Frags f0, f1;
        fetch(f0, ac, bc, 0);
        stage_a(an);
        dma_b(bn);
        load_a();
        fetch(f1, ac, bc, 1);
        acc.multiply(f0);
        acc.multiply(f1);
    };
    if (n <= 0 || range >= g.ranges) return;  // uniform (ranges <= units and grid = ranges x tiles_n: does not occur)
    load_a();
    dma_b(b0);
    stage_a(a0);
    load_a();
    int left = n, c_pr = p0 - tile0 * g.pairs;
    for (int t = tile0; left > 0; ++t, c_pr = 0) {  // the range's tile rows
        const int here = min(g.pairs - c_pr, left);
        acc.clear();
        for (int j = 0; j < here; ++j) {
            slice(a0, b0, a1, b1);
            slice(a1, b1, a0, b0);
        }
        flush(t);
        left -= here;
    }
    // no transfer into LDS outlives the workgroup
    stage_barrier<0>();
}

// C = the sum of each tile's parts in order, times the row's (ri) or the
// common factor.  A lane takes one 16-byte unit of the parts: four consecutive
// rows of a column, 32 lanes 32 columns.
template <bool TA>
__global__ __launch_bounds__(256) void h2_reduce_kernel(H2Args g, const float *__restrict__ ri,
                                                        const float *__restrict__ common, float *__restrict__ C) {
    constexpr int kUnits = T * T / 4;
    const int tile = static_cast<int>(blockIdx.x) / (kUnits / 256);
    const int unit = (static_cast<int>(blockIdx.x) % (kUnits / 256)) * 256 + threadIdx.x;
    const int tm = tile / g.tiles_n, tn = tile - tm * g.tiles_n;
    const int64_t ub = static_cast<int64_t>(tm) * g.pairs;
    const int parts = h2_owner(ub + g.pairs - 1, g.units, g.ranges) - h2_owner(ub, g.units, g.ranges) + 1;
    const f32x4 *W = reinterpret_cast<const f32x4 *>(g.ws) + static_cast<uint64_t>(tile) * g.maxparts * kUnits + unit;
    const int lane = unit & 63, q = (unit >> 6) & 3, jj = (unit >> 8) & 1, i = (unit >> 9) & 1, wave = unit >> 10;
    const int gi = tm * T + (wave >> 1) * 64 + 32 * i + 8 * q + 4 * (lane >> 5);
    const int gj = tn * T + (wave & 1) * 64 + 32 * jj + (lane & 31);
    if (gi >= g.M || gj >= g.N) return;
    f32x4 s = W[0];
#pragma unroll 4
    for (int p = 1; p < parts; ++p) s += W[static_cast<uint64_t>(p) * kUnits];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        const int r = gi + e;
        if (r < g.M) C[static_cast<uint64_t>(r) * g.N + gj] = s[e] * (TA ? *common : ri[r]);
    }
}

struct H2Plan {
    int tiles_m, tiles_n, pairs, units, ranges, maxparts;
    uint64_t bytes;  // partial tiles
};

// Two workgroups per CU share the slices, unless that leaves a workgroup
// fewer than two pairs of them (128 k): the parts' traffic and the serial sum
// of a tile's parts then cost more than the idle CUs (512 x 1024, rank 64:
// 488 us a round trip with two, 494 with one and 508 with four).
H2Plan h2_plan(int M, int N, int K) {
    H2Plan p{};
    p.tiles_m = static_cast<int>(ceil_div(M, T));
    p.tiles_n = static_cast<int>(ceil_div(N, T));
    p.pairs = static_cast<int>(ceil_div(K, 2 * BK));
    p.units = p.tiles_m * p.pairs;
    const int most = std::max(1, 2 * cu_count() / p.tiles_n);
    p.ranges = std::max(1, std::min({most, std::max(p.tiles_m, p.units / 2), p.units}));
    p.maxparts = 1;
    for (int t = 0; t < p.tiles_m; ++t) {
        const int64_t b = static_cast<int64_t>(t) * p.pairs;
        p.maxparts =
            std::max(p.maxparts, h2_owner(b + p.pairs - 1, p.units, p.ranges) - h2_owner(b, p.units, p.ranges) + 1);
    }
    p.bytes = static_cast<uint64_t>(p.tiles_m) * p.tiles_n * p.maxparts * T * T * sizeof(float);
    return p;
}

int pad64(int n) { return static_cast<int>(ceil_div(n, 64) * 64); }

}  // namespace

// Bytes of the partial tiles of an M x N x K product.
uint64_t h2_workspace_bytes(int M, int N, int K) { return h2_plan(M, N, K).bytes; }

// f16 values of the two planes of a K x N operand B.
uint64_t h2_plane_units(int K, int N) { return 2 * static_cast<uint64_t>(pad64(K)) * pad64(N); }

bool h2_supported(int K) { return K >= 2 * BK; }

void launch_h2_scales(const float *A, int m, int n, const H2Scales &s, float *R, uint64_t fill, uint64_t seed,
                      hipStream_t stream) {
    BSQ_REQUIRE(A && m > 0 && n > 0 && s.exponent && s.scale && s.inverse && (R || fill == 0),
                "h2 scales: bad arguments");
    const uint64_t draws = std::min<uint64_t>(ceil_div(fill, 4 * kThreads), static_cast<uint64_t>(cu_count()) * 8);
    row_scale_kernel<<<static_cast<unsigned>(m + draws), kThreads, 0, stream>>>(A, m, n, s.exponent, s.scale,
                                                                               s.inverse, R, fill, seed);
    BSQ_HIP(hipGetLastError());
}

H2Planes h2_planes(bool ta, int K, int q, const H2Scales &s, uint16_t *planes) {
    H2Planes b;
    b.K = K;
    b.rows = pad64(K);
    b.rot = ta ? 0 : -K & 7;
    b.np = pad64(q);
    b.hi = planes;
    b.lo = planes + static_cast<uint64_t>(b.rows) * b.np;
    b.exponent = ta ? s.exponent : nullptr;
    b.emax = s.emax;
    return b;
}

void launch_h2_split(const float *B, int q, const H2Planes &b, const H2Scales &s, int new_rows, hipStream_t stream) {
    BSQ_REQUIRE(q > 0 && (B || b.rows == 0) && s.emax && s.common, "h2 split: bad arguments");
    const uint64_t units = static_cast<uint64_t>(b.rows / 8) * b.np;
    if (units == 0 && new_rows == 0) return;
    split_b_kernel<<<static_cast<unsigned>(std::max<uint64_t>(1, ceil_div(units, kThreads))), kThreads, 0, stream>>>(
        B, b.K, q, b.np, b.rows / 8, b.rot, s.exponent, new_rows, b.exponent != nullptr, s.emax, s.common,
        reinterpret_cast<u32x4 *>(b.hi), reinterpret_cast<u32x4 *>(b.lo));
    BSQ_HIP(hipGetLastError());
}

void launch_h2_gemm(bool ta, int m, int n, int q, const float *A, const H2Scales &s, const H2Planes &b, float *C,
                    float *workspace, uint64_t workspace_bytes, hipStream_t stream) {
    const int M = ta ? n : m, K = ta ? m : n;
    BSQ_REQUIRE(M > 0 && q > 0 && h2_supported(K) && A && C && b.hi && workspace, "h2 gemm: bad arguments");
    const H2Plan p = h2_plan(M, q, K);
    BSQ_REQUIRE(p.bytes <= workspace_bytes, "h2 gemm: workspace too small");
    H2Args g{};
    BSQ_REQUIRE(b.K == K && b.np == pad64(q), "h2 gemm: planes of another operand");
    g.A = A;
    g.bh = reinterpret_cast<const u32x4 *>(b.hi);
    g.bl = reinterpret_cast<const u32x4 *>(b.lo);
    g.rs = s.scale;
    g.ws = workspace;
    g.M = M;
    g.N = q;
    g.K = K;
    g.lda = n;
    g.np = b.np;
    g.tiles_n = p.tiles_n;
    g.pairs = p.pairs;
    g.units = p.units;
    g.ranges = p.ranges;
    g.maxparts = p.maxparts;
    const dim3 grid(static_cast<unsigned>(p.ranges * p.tiles_n)),
        rgrid(static_cast<unsigned>(p.tiles_m * p.tiles_n * (T * T / 4 / 256)));
    if (ta) gemm_h2_kernel<true><<<grid, kThreads, 0, stream>>>(g);
    else gemm_h2_kernel<false><<<grid, kThreads, 0, stream>>>(g);
    BSQ_HIP(hipGetLastError());
    if (ta) h2_reduce_kernel<true><<<rgrid, 256, 0, stream>>>(g, nullptr, s.common, C);
    else h2_reduce_kernel<false><<<rgrid, 256, 0, stream>>>(g, s.inverse, nullptr, C);
    BSQ_HIP(hipGetLastError());
}

}  // namespace bsq
