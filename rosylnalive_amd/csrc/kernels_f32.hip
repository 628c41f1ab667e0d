// The float32 contractions of the reference catalog (matmul_bf16w, attention_gqa_causal) on gfx950's f32 matrix cores.
//
// CpuRef F32 defines every contraction as one chain of fused multiply-adds in increasing k from +0. The f32 MFMAs do
// exactly that: v_mfma_f32_16x16x4_f32 returns fma(a3, b3, fma(a2, b2, fma(a1, b1, fma(a0, b0, c)))) bit for bit
// (measured against fmaf on 2^20 outputs for each of: uniform values, 40 binades, products and sums in the denormal
// range, denormal inputs, arbitrary bit patterns). So the kernels below keep the reference's bits at 148 TFLOP/s peak
// (v_fma_f32: 62).
//
// Built with -ffp-contract=off, as kernels_catalog.hip.
#include "kernels_f32.hpp"

#include "fast_common.hpp"

namespace lrm {
namespace f32k {

using fast::f32x4;
using fast::lds_barrier;
using fast::u32x4;
typedef float f32x2 __attribute__((ext_vector_type(2)));

// ---------------------------------------------------------------- matmul_bf16w
// An output is one chain of k / 4 dependent MFMAs (32 cycles each, 8 per k: what dependent v_fma_f32 take, too), so a
// wave with one tile must issue its MFMAs back to back. It may issue LDS reads between them for nothing, but every VALU
// instruction between two dependent MFMAs adds its 4 cycles and every interruption about 8 more (measured: 33 cycles per
// MFMA alone, 45 with one VALU instruction between, 57 with four; a loop that also widened, staged and addressed took
// 1170 cycles per 64 k instead of 512). So half of a block's waves only stage: they load x and w (16 bytes per lane, D
// tiles in flight), widen w and write both to LDS; the others only read operands and multiply. One barrier per tile; the
// operands of tile t + 1 are read while tile t multiplies and tile t + 2 is stored, NB LDS stages. Against 16 x 64 tiles on
// the vector ALUs: 29 matmuls of a decode step (0.6B, four layers) 142 us each, the 15 of a 150-row forward 146 us each;
// here 5.8 us for k 1024 at one row, 17.5 at 150 rows.
//
// The operand of step s of a 16x16x4 MFMA holds k = 4 s + g in lane group g = lane / 16, so a staged tile is kept by
// group, [g][row][k / 4]: one 16-byte LDS read gives a lane four consecutive steps. Rows are KS / 4 + 4 words and a
// group's plane a multiple of 64: such a read takes 4.2 cycles a wave (rows of KS + 4 words holding all four groups: 8).

// k at or past the end: x = +0 and w = -0, whose product -0 leaves every chain value as it is, -0 included.
constexpr uint32_t kNegZeroPair = 0x80008000u;

// A block computes a (16 WR TM) x (16 WC TN) tile: WR x WC multiplying waves of TM x TN MFMA tiles, as many staging
// waves, in groups of D tiles of KS along k.
// VEC: x and w 16-byte aligned, k a multiple of 8; otherwise element loads. END, where k ends: FULL, with a group, no padding;
// GROUPS, anywhere, tiles past k multiply the padding; TILES, with the tile that holds the last of k. TILES is for k up to 512
// (32-row tiles) or 384, where a group is most of the work (padded to groups, 17 to 150 rows of k 64 took 6.4 us against 2.8,
// of 129 10.4 against 5.0); past that, its branches cost more than the padding (1 x 64 x 504 4.4 us in groups, 4.8 in tiles;
// 1 x 20,000 x 1000 16.0 and 24.5).
enum class End { FULL, GROUPS, TILES };
// Up to three weights over one x share a launch, their column tiles side by side: a decode step's q, k and v projections
// are 64 to 128 chains' worth of blocks each, and one after another each waits its chain out on an idle chip.
template <int WR, int WC, int TM, int TN, int KS, int D, int NB, bool VEC, End END>
__global__ __launch_bounds__(128 * WR * WC) void k_matmul_mfma(const float* __restrict__ x, MatmulGroup group,
                                                               uint32_t m, uint32_t k) {
    constexpr int BM = 16 * WR * TM, BN = 16 * WC * TN, NT = 64 * WR * WC, STEPS = KS / 4, ROW = STEPS + 4;
    constexpr bool FULL = END == End::FULL, TILES = END == End::TILES;
    constexpr int XR = NT / (KS / 4), WRW = NT / (KS / 8);  // rows staged per pass
    constexpr int XQ = BM / XR, WQ = BN / WRW;              // 16-byte chunks per staging thread
    static_assert(XQ >= 1 && WQ >= 1 && BM % XR == 0 && BN % WRW == 0, "whole chunks");
    static_assert(D % NB == 0 && NB >= 3 && D % 2 == 0, "stages and operand sets of the unrolled loop");
    static_assert(KS == 64, "chunk maps");
    __shared__ float xs[NB][4 * BM * ROW];
    __shared__ float ws[NB][4 * BN * ROW];
    uint32_t part = 0, bx = blockIdx.x;
    while (part + 1 < group.count && bx >= (group.n[part] + BN - 1) / BN) bx -= (group.n[part++] + BN - 1) / BN;
    const uint16_t* __restrict__ w = group.w[part];
    float* __restrict__ y = group.y[part];
    const uint32_t n = group.n[part], i0 = blockIdx.y * BM, j0 = bx * BN;
    if (threadIdx.x >= NT) {
        const uint32_t t = threadIdx.x - NT;
        // chunk q of this thread: x row xr0 + XR q, k 4 xc ..; w row wr0 + WRW q, k 8 wcx ..; the rows a store touches
        // at once lie four apart (distinct banks)
        const uint32_t xc = t & (KS / 4 - 1), wcx = t & (KS / 8 - 1);
        const uint32_t xr0 = ((t >> 4) & 3u) * (XR / 4) + (t >> 6);
        const uint32_t wr0 = NT >= 128
                                 ? ((t >> 3) & 3u) * 4u + ((t >> 5) & 1u) + ((t >> 6) & 1u) * 2u + (t >> 7) * 16u
                                 : t / (KS / 8);
        u32x4 xreg[D][XQ], wreg[D][WQ];
        // FULL: buffer loads, the k offset in a scalar register. A VALU instruction of this wave also delays the
        // multiplying wave of its SIMD, and 64-bit addresses took most of them.
        const uint32_t xrows = m - i0 < uint32_t(BM) ? m - i0 : uint32_t(BM);
        const uint32_t wrows = n - j0 < uint32_t(BN) ? n - j0 : uint32_t(BN);
        const auto xrsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(x + size_t(i0) * k), (short)0,
                                                             int(xrows * k * 4u), 0x00020000);
        const auto wrsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(w + size_t(j0) * k), (short)0,
                                                             int(wrows * k * 2u), 0x00020000);
        uint32_t xo[XQ], wo[WQ];
#pragma unroll
        for (int q = 0; q < XQ; ++q) xo[q] = (xr0 + XR * q < xrows ? xr0 + XR * q : xrows - 1u) * k * 4u + 16u * xc;
#pragma unroll
        for (int q = 0; q < WQ; ++q) wo[q] = (wr0 + WRW * q < wrows ? wr0 + WRW * q : wrows - 1u) * k * 2u + 16u * wcx;
        auto load = [&](int d, uint32_t k0) {
            if constexpr (FULL) {
                const uint32_t ks = k0 < k ? k0 : k - KS;  // (a tile past the last: the last, never multiplied)
#pragma unroll
                for (int q = 0; q < XQ; ++q) xreg[d][q] = __builtin_amdgcn_raw_buffer_load_b128(xrsrc, xo[q], ks * 4u, 0);
#pragma unroll
                for (int q = 0; q < WQ; ++q) wreg[d][q] = __builtin_amdgcn_raw_buffer_load_b128(wrsrc, wo[q], ks * 2u, 0);
                __builtin_amdgcn_sched_barrier(0);
                return;
            }
#pragma unroll
            for (int q = 0; q < XQ; ++q) {
                uint32_t row = i0 + xr0 + XR * q;
                row = row < m ? row : m - 1u;
                const uint32_t kk = k0 + 4u * xc;
                if constexpr (VEC) {
                    xreg[d][q] = *reinterpret_cast<const u32x4*>(x + size_t(row) * k + (kk < k ? kk : 0u));
                } else {
#pragma unroll
                    for (uint32_t e = 0; e < 4; ++e)
                        xreg[d][q][e] = __float_as_uint(x[size_t(row) * k + (kk + e < k ? kk + e : 0u)]);
                }
            }
#pragma unroll
            for (int q = 0; q < WQ; ++q) {
                uint32_t col = j0 + wr0 + WRW * q;
                col = col < n ? col : n - 1u;
                const uint32_t kk = k0 + 8u * wcx;
                if constexpr (VEC) {
                    wreg[d][q] = *reinterpret_cast<const u32x4*>(w + size_t(col) * k + (kk < k ? kk : 0u));
                } else {
#pragma unroll
                    for (uint32_t e = 0; e < 4; ++e) {
                        const uint32_t a = kk + 2u * e, b = a + 1u;
                        const uint32_t lo = w[size_t(col) * k + (a < k ? a : 0u)],
                                       hi = w[size_t(col) * k + (b < k ? b : 0u)];
                        wreg[d][q][e] = (a < k ? lo : 0x8000u) | (b < k ? hi << 16 : 0x80000000u);
                    }
                }
            }
            __builtin_amdgcn_sched_barrier(0);
        };
        auto store = [&](int d, uint32_t k0) {  // set d's tile (at k0) to LDS stage d % NB
#pragma unroll
            for (int q = 0; q < XQ; ++q) {
                const uint32_t kk = k0 + 4u * xc;
                float* p = &xs[d % NB][(xr0 + XR * q) * ROW + xc];
#pragma unroll
                for (uint32_t g = 0; g < 4; ++g) {
                    const bool in = FULL || (VEC ? kk < k : kk + g < k);
                    p[g * BM * ROW] = in ? __uint_as_float(xreg[d][q][g]) : 0.f;
                }
            }
#pragma unroll
            for (int q = 0; q < WQ; ++q) {
                u32x4 v = wreg[d][q];
                if (VEC && !FULL && k0 + 8u * wcx >= k) v = u32x4{kNegZeroPair, kNegZeroPair, kNegZeroPair, kNegZeroPair};
                float* p = &ws[d % NB][(wr0 + WRW * q) * ROW + 2 * wcx];
#pragma unroll
                for (int g = 0; g < 4; ++g) {  // k 8 wcx + g and + 4 + g
                    const uint32_t a = v[g >> 1], b = v[2 + (g >> 1)];
                    f32x2 pair;
                    pair[0] = __uint_as_float((g & 1) ? a & 0xFFFF0000u : a << 16);
                    pair[1] = __uint_as_float((g & 1) ? b & 0xFFFF0000u : b << 16);
                    *reinterpret_cast<f32x2*>(p + g * BN * ROW) = pair;
                }
            }
            __builtin_amdgcn_sched_barrier(0);
        };
        auto holds = [&](uint32_t k0) { return !TILES || k0 < k; };  // a tile at k0 is loaded and stored
#pragma unroll
        for (int d = 0; d < D; ++d)
            if (holds(uint32_t(d) * KS)) load(d, uint32_t(d) * KS);
        store(0, 0);
        if (holds(KS)) store(1, KS);
        lds_barrier();
        uint32_t k0 = 0;
        do {  // (at least once: a loop that may not run lets the compiler sink the first loads past the barrier above)
#pragma unroll
            for (int d = 0; d < D; ++d) {
                if (holds(k0 + uint32_t(d + D) * KS)) load(d, k0 + uint32_t(d + D) * KS);  // this set's tile is in LDS
                if (holds(k0 + uint32_t(d + 2) * KS)) store((d + 2) % D, k0 + uint32_t(d + 2) * KS);
                lds_barrier();
                if (!holds(k0 + uint32_t(d + 1) * KS)) break;
            }
            k0 += D * KS;
        } while (k0 < k);
        return;
    }
    const uint32_t lane = threadIdx.x & 63u, wv = threadIdx.x >> 6, wr = wv / WC, wc = wv % WC;
    const uint32_t r16 = lane & 15u, grp = lane >> 4;
    const uint32_t xoff = (grp * BM + wr * TM * 16u + r16) * ROW, woff = (grp * BN + wc * TN * 16u + r16) * ROW;
    f32x4 acc[TM][TN], av[2][TM][STEPS / 4], bv[2][TN][STEPS / 4];
#pragma unroll
    for (int a = 0; a < TM; ++a)
#pragma unroll
        for (int b = 0; b < TN; ++b) acc[a][b] = f32x4{0.f, 0.f, 0.f, 0.f};
    auto read = [&](int set, int d) {
#pragma unroll
        for (int q = 0; q < STEPS / 4; ++q) {
#pragma unroll
            for (int a = 0; a < TM; ++a)
                av[set][a][q] = *reinterpret_cast<const f32x4*>(&xs[d % NB][xoff + a * 16 * ROW + 4 * q]);
#pragma unroll
            for (int b = 0; b < TN; ++b)
                bv[set][b][q] = *reinterpret_cast<const f32x4*>(&ws[d % NB][woff + b * 16 * ROW + 4 * q]);
        }
        __builtin_amdgcn_sched_barrier(0);
    };
    lds_barrier();
    read(0, 0);
    uint32_t k0 = 0;
    do {
#pragma unroll
        for (int d = 0; d < D; ++d) {
            read((d + 1) & 1, d + 1);
#pragma unroll
            for (int q = 0; q < STEPS / 4; ++q)
#pragma unroll
                for (int i = 0; i < 4; ++i)
#pragma unroll
                    for (int a = 0; a < TM; ++a)
#pragma unroll
                        for (int b = 0; b < TN; ++b)
                            acc[a][b] = __builtin_amdgcn_mfma_f32_16x16x4f32(av[d & 1][a][q][i], bv[d & 1][b][q][i],
                                                                             acc[a][b], 0, 0, 0);
            __builtin_amdgcn_sched_barrier(0);
            lds_barrier();
            if (TILES && k0 + uint32_t(d + 1) * KS >= k) break;  // (with the staging waves)
        }
        k0 += D * KS;
    } while (k0 < k);
#pragma unroll
    for (int a = 0; a < TM; ++a)
#pragma unroll
        for (int b = 0; b < TN; ++b) {
            const uint32_t j = j0 + (wc * TN + b) * 16u + r16;
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const uint32_t i = i0 + (wr * TM + a) * 16u + grp * 4u + r;
                if (i < m && j < n) y[size_t(i) * n + j] = acc[a][b][r];
            }
        }
}

static bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }

template <int WR, int WC, int TM, int TN, int KS, int D, int NB>
static void launch_mfma(bool vec, const float* x, const MatmulGroup& g, uint32_t m, uint32_t k, hipStream_t s) {
    constexpr uint32_t BM = 16 * WR * TM, BN = 16 * WC * TN;
    uint32_t tiles = 0;
    for (uint32_t i = 0; i < g.count; ++i) tiles += (g.n[i] + BN - 1) / BN;
    const dim3 grid(tiles, (m + BM - 1) / BM), block(128 * WR * WC);
    constexpr uint32_t kTilesTo = BM == 32 ? 512 : 384;
    auto go = [&](auto kernel) { hipLaunchKernelGGL(kernel, grid, block, 0, s, x, g, m, k); };
    if (vec && k % (D * KS) == 0 && uint64_t(k) * (BM > BN / 2 ? BM : BN / 2) * 4 < (1ull << 31))
        go(k_matmul_mfma<WR, WC, TM, TN, KS, D, NB, true, End::FULL>);
    else if (vec && k <= kTilesTo)
        go(k_matmul_mfma<WR, WC, TM, TN, KS, D, NB, true, End::TILES>);
    else if (vec)
        go(k_matmul_mfma<WR, WC, TM, TN, KS, D, NB, true, End::GROUPS>);
    else if (k <= kTilesTo)
        go(k_matmul_mfma<WR, WC, TM, TN, KS, D, NB, false, End::TILES>);
    else
        go(k_matmul_mfma<WR, WC, TM, TN, KS, D, NB, false, End::GROUPS>);
}

// k = 0: every output is an empty chain, +0. The tile kernels read element 0 of every row, which does not exist then.
__global__ __launch_bounds__(256) void k_zero_rows(MatmulGroup group, uint32_t m) {
    for (uint32_t i = 0; i < group.count; ++i) {
        const uint64_t n = uint64_t(m) * group.n[i], step = uint64_t(gridDim.x) * 256u;
        for (uint64_t e = uint64_t(blockIdx.x) * 256u + threadIdx.x; e < n; e += step) group.y[i][e] = 0.f;
    }
}

// Short k, where staging through registers in groups is most of the tile kernels' time: a 16 x 64 tile per block on the
// vector ALUs, thread t column t % 64 of rows 4 (t / 64) .., K of k staged at a time.
template <uint32_t K>
__global__ __launch_bounds__(256) void k_matmul_short(const float* __restrict__ x, MatmulGroup group, uint32_t m, uint32_t k) {
    __shared__ float xs[16][K];
    __shared__ float ws[64][K + 1];
    uint32_t part = 0, bx = blockIdx.x;
    while (part + 1 < group.count && bx >= (group.n[part] + 63u) / 64u) bx -= (group.n[part++] + 63u) / 64u;
    const uint16_t* __restrict__ w = group.w[part];
    const uint32_t t = threadIdx.x, n = group.n[part], i0 = blockIdx.y * 16u, j0 = bx * 64u, col = t % 64u, r0 = t / 64u * 4u;
    const uint32_t rows = m - i0 < 16u ? m - i0 : 16u, cols = n - j0 < 64u ? n - j0 : 64u;
    float acc[4] = {0.f, 0.f, 0.f, 0.f};
    for (uint32_t p0 = 0; p0 < k; p0 += K) {
        const uint32_t ks = k - p0 < K ? k - p0 : K;
        if (p0) __syncthreads();
#pragma unroll
        for (uint32_t e = t; e < 16u * K; e += 256u)
            if (e / K < rows && e % K < ks) xs[e / K][e % K] = x[size_t(i0 + e / K) * k + p0 + e % K];
#pragma unroll
        for (uint32_t e = t; e < 64u * K; e += 256u)
            if (e / K < cols && e % K < ks)
                ws[e / K][e % K] = __uint_as_float(uint32_t(w[size_t(j0 + e / K) * k + p0 + e % K]) << 16);
        __syncthreads();
        for (uint32_t p = 0; p < ks; ++p) {
            const float wv = ws[col][p];  // (columns past n, rows past m: never stored)
#pragma unroll
            for (uint32_t r = 0; r < 4; ++r) acc[r] = fmaf(xs[r0 + r][p], wv, acc[r]);
        }
    }
    if (col >= cols) return;
#pragma unroll
    for (uint32_t r = 0; r < 4; ++r)
        if (r0 + r < rows) group.y[part][size_t(i0 + r0 + r) * n + j0 + col] = acc[r];
}

void matmul_bf16w(const float* x, const MatmulGroup& g, uint32_t m, uint32_t k, hipStream_t s) {
    if (k == 0) {
        uint64_t most = 0;
        for (uint32_t i = 0; i < g.count; ++i) most = most > g.n[i] ? most : g.n[i];
        const uint64_t blocks = (most * m + 255) / 256;
        hipLaunchKernelGGL(k_zero_rows, dim3(uint32_t(blocks < 4096 ? blocks : 4096)), dim3(256), 0, s, g, m);
        return;
    }
    bool vec = k % 8 == 0 && aligned16(x);
    uint64_t n = 0, big = 0, small = 0;
    for (uint32_t i = 0; i < g.count; ++i) {
        vec = vec && aligned16(g.w[i]);
        n += g.n[i];
        big += uint64_t((m + 63) / 64) * ((g.n[i] + 63) / 64);
        small += uint64_t((m + 31) / 32) * ((g.n[i] + 31) / 32);
    }
    // The short kernel up to k 32, and further where the tile kernels' blocks, of few rows or columns and 60 KB and more of
    // LDS, need many rounds of the chip. Short kernel against tile kernels, us: 17 x 1024 x 16 3.1 / 2.7, 150 x 4096 x 16 3.7 /
    // 4.5, 150 x 20,000 x 16 7.6 / 13.2, x 33 14.9 / 21.4, 1 x 20,000 x 16 3.1 / 3.8, 1 x 100,000 x 33 7.5 / 12.8, x 64 9.6 /
    // 10.6, x 129 25.2 / 31.4; but 17 x 1024 x 33 5.3 / 3.1.
    const bool wide = (big + 255) / 256 * 800 < small, many = m <= 16 ? n > 65536 : !wide && small > 1024;
    if (k <= (!many ? 32u : m <= 16 ? (vec ? 80u : 320u) : (vec ? 32u : 128u))) {
        uint32_t tiles = 0;
        for (uint32_t i = 0; i < g.count; ++i) tiles += (g.n[i] + 63) / 64;
        auto go = [&](auto kernel) { hipLaunchKernelGGL(kernel, dim3(tiles, (m + 15) / 16), dim3(256), 0, s, x, g, m, k); };
        if (k <= 16) return go(k_matmul_short<16>);
        return k <= 32 ? go(k_matmul_short<32>) : go(k_matmul_short<64>);
    }
    // Up to 16 rows one MFMA tile per block: an output is one chain however many columns a block has, and two waves find
    // SIMDs of their own (1 x 1024 x 1024: 5.8 us; 32-column blocks 6.0); past 16,384 columns, where the weights' stream
    // counts, 32 columns (1 x 151,936 x 1024: 79.7 us against 84.1). Above: 32 x 32 tiles, about 26 ns a tile at k 1024
    // however they fill the chip (480 tiles 14.7 us, 960 26.3, 6144 139), or 64 x 64, 21 us a round of 256 (240 tiles 23.2
    // us, 480 42.8, 1536 126): the larger where its rounds take less (a round for 800 small tiles).
    if (m <= 16 && n <= 16384)
        launch_mfma<1, 1, 1, 1, 64, 4, 4>(vec, x, g, m, k, s);
    else if (m <= 16)
        launch_mfma<1, 2, 1, 1, 64, 8, 4>(vec, x, g, m, k, s);
    else if (wide)
        launch_mfma<2, 2, 2, 2, 64, 4, 4>(vec, x, g, m, k, s);
    else
        launch_mfma<2, 2, 1, 1, 64, 8, 4>(vec, x, g, m, k, s);
}

// ---------------------------------------------------------------- attention_gqa_causal
// The reference's arithmetic (kernels_catalog.hip, k_attention_f32): 64-key blocks, a fused dot in increasing d, online
// softmax per block with weights against the running maximum, block sums in increasing key from +0, then
// l = fma(l, alpha, sum), o = fma(o, alpha, value). All of it maps onto MFMA chains with the same bits:
// S^T = K Q^T, the block sum as a row of ones times P^T, O^T = V^T P^T.
//
// A tile is 16 columns = 16 (query row, query head) pairs of one KV head (head fastest), so heads that share K/V share
// the loads. S^T leaves key 16 t + 4 (lane / 16) + r of column lane % 16 in register r; the P^T operand of step s wants
// key 4 s + lane / 16: one 4 x 4 exchange between lane groups (two permlane32 and two permlane16 swaps per 16 keys).
// K and Q operands come from 16-byte loads through the same exchange; V operands are 16-byte loads whose four elements
// feed four tiles (tile (c, e) row i = dimension 16 E c + E i + e). No LDS for operands.
//
// W waves share a tile's keys, wave w taking block w of each group of W: the blocks' scores, sums and values do not
// depend on each other given the running maxima, which every wave forms from the blocks' maxima in order; the ordered
// combine of o is split over the waves. W = 1: four tiles per workgroup, no sharing.
// Bound by each block's chains (128 dimensions: 32 dependent MFMAs per 16 keys for the scores, 16 for the values) and by
// the K and V loads of a workgroup's CU. 16 heads, 8 KV heads, 150 rows: 156.6 us on the vector ALUs, 19.1 here.

// out i of lane group g = in g of lane group i
__device__ __forceinline__ void transpose4(float (&v)[4]) {
    uint32_t a = __float_as_uint(v[0]), b = __float_as_uint(v[1]), c = __float_as_uint(v[2]), d = __float_as_uint(v[3]);
    const auto ac = __builtin_amdgcn_permlane32_swap(a, c, false, false);
    const auto bd = __builtin_amdgcn_permlane32_swap(b, d, false, false);
    const auto lo = __builtin_amdgcn_permlane16_swap(ac[0], bd[0], false, false);
    const auto hi = __builtin_amdgcn_permlane16_swap(ac[1], bd[1], false, false);
    v[0] = __uint_as_float(lo[0]);
    v[1] = __uint_as_float(lo[1]);
    v[2] = __uint_as_float(hi[0]);
    v[3] = __uint_as_float(hi[1]);
}

template <int HD, int W>
__global__ __launch_bounds__(W == 1 ? 256 : 64 * W) void k_attention_mfma(
    const float* __restrict__ q, const float* __restrict__ kc, const float* __restrict__ vc, float* __restrict__ y,
    uint32_t rows, uint32_t q_row0, uint32_t past, uint32_t qh, uint32_t kvh, float scale) {
    constexpr int E = HD % 64 == 0 ? 4 : 1, NC = HD / (16 * E), U = HD / 16;
    constexpr int REGS = HD / 4;  // O registers per lane: 16 columns x HD over 64 lanes
    const uint32_t lane = threadIdx.x & 63u, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t col = lane & 15u, grp = lane >> 4;
    const uint32_t group = qh / kvh, total = rows * group, tiles = (total + 15u) / 16u;
    // the longest first; W = 1, where workgroups wait for their turn, over all KV heads (one dimension: head fastest)
    const uint32_t kvhead = W == 1 ? blockIdx.x % kvh : blockIdx.y;
    const uint32_t tb = W == 1 ? blockIdx.x / kvh * 4u + wv : blockIdx.x;
    if (tb >= tiles) return;
    const uint32_t tile = tiles - 1u - tb;
    const uint32_t raw = tile * 16u + col, idx = raw < total ? raw : total - 1u;
    const uint32_t row = idx / group, head = kvhead * group + idx % group;
    const uint32_t keys = past + row + 1u;                       // this column's
    const uint32_t first_keys = past + tile * 16u / group + 1u;  // the tile's fewest
    const uint32_t last_idx = tile * 16u + 15u < total ? tile * 16u + 15u : total - 1u;
    const uint32_t max_keys = past + last_idx / group + 1u;
    const uint32_t nblocks = (max_keys + 63u) / 64u;
    const size_t kv_stride = size_t(kvh) * HD;
    const float* kb = kc + size_t(kvhead) * HD + 4u * grp;
    const float* vb = vc + size_t(kvhead) * HD + E * col;
    const size_t qoff = (size_t(q_row0 + row) * qh + head) * HD;

    float qf[U][4];
    // A block's K and V come in whole: all loads in flight at once (the compiler, left alone, keeps a few), V's while
    // the scores' maxima meet, the next block's K while the values are combined.
    auto load_k = [&](uint32_t b, f32x4 (&kr)[U][4]) {
        const float* p[4];
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            const uint32_t j = b * 64u + 16u * t + col;
            p[t] = kb + size_t(j < max_keys ? j : max_keys - 1u) * kv_stride;
        }
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
            for (int t = 0; t < 4; ++t) kr[u][t] = *reinterpret_cast<const f32x4*>(p[t] + 16 * u);
        __builtin_amdgcn_sched_barrier(0);
    };
    // E values of each tile group c at step st: key 64 b + 4 st + grp (a key past the tile's last: its last)
    auto load_v = [&](uint32_t b, float (&vr)[16][NC][E]) {
#pragma unroll
        for (int st = 0; st < 16; ++st) {
            const uint32_t j = b * 64u + 4u * st + grp;
            const float* p = vb + size_t(j < max_keys ? j : max_keys - 1u) * kv_stride;
#pragma unroll
            for (int c = 0; c < NC; ++c) {
                if constexpr (E == 4) {
                    const f32x4 x = *reinterpret_cast<const f32x4*>(p + 64 * c);
#pragma unroll
                    for (int e = 0; e < 4; ++e) vr[st][c][e] = x[e];
                } else {
                    vr[st][c][0] = p[16 * c];
                }
            }
        }
        __builtin_amdgcn_sched_barrier(0);
    };
    // scores of block b: s[t][r] = key 64 b + 16 t + 4 grp + r (times scale); returns the block's maximum over this
    // column's keys (-inf for none)
    auto score = [&](uint32_t b, const f32x4 (&kr)[U][4], f32x4 (&s)[4]) {
        float mx = -INFINITY;
#pragma unroll
        for (int t = 0; t < 4; ++t) s[t] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int u = 0; u < U; ++u) {
            float kf[4][4];
#pragma unroll
            for (int t = 0; t < 4; ++t) {
#pragma unroll
                for (int i = 0; i < 4; ++i) kf[t][i] = kr[u][t][i];
                transpose4(kf[t]);
            }
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int t = 0; t < 4; ++t) s[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(kf[t][i], qf[u][i], s[t], 0, 0, 0);
        }
#pragma unroll
        for (int t = 0; t < 4; ++t) {
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                // a key past the column's own scores -inf: weight 0 (or NaN where every score is -inf or NaN, and the
                // reference's weights are NaN too)
                s[t][r] = b * 64u + 16u * t + 4u * grp + r < keys ? s[t][r] * scale : -INFINITY;
                mx = fmaxf(mx, s[t][r]);
            }
        }
        return fast::cross_rows_max(mx);
    };

    // the block's values and sum against the maximum mn: acc (register (c, e, r) = dimension 16 E c + E (4 grp + r) + e
    // of this column), bs the sum of the weights
    auto values = [&](uint32_t b, const f32x4 (&s)[4], float mn, const float (&vr)[16][NC][E], f32x4 (&acc)[NC][E],
                      float& bs) {
        float pf[4][4];
#pragma unroll
        for (int t = 0; t < 4; ++t) {
#pragma unroll
            for (int r = 0; r < 4; ++r) pf[t][r] = expf(s[t][r] - mn);
            transpose4(pf[t]);
        }
        f32x4 sum = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int st = 0; st < 16; ++st) sum = __builtin_amdgcn_mfma_f32_16x16x4f32(1.f, pf[st >> 2][st & 3], sum, 0, 0, 0);
        bs = sum[0];
        // A key past a column's own has weight 0, and its product is a zero of its value's sign: it leaves the chain as it is
        // while the value is finite and the chain is not -0 (a chain of products that underflow). Where a block with such
        // keys holds an infinity or a NaN, or ends at a zero, each column runs alone with those values at -0 (a product of
        // -0 changes no chain). The look at the ends costs 512 rows of 16 heads 52.0 -> 54.1 us.
        const bool partial = b * 64u + 64u > first_keys;
        bool odd = false;
        if (partial) {
            float bad = 0.f;  // NaN once a value is not finite
#pragma unroll
            for (int st = 0; st < 16; ++st)
#pragma unroll
                for (int c = 0; c < NC; ++c)
#pragma unroll
                    for (int e = 0; e < E; ++e) bad = fmaf(vr[st][c][e], 0.f, bad);
            odd = __ballot(bad != bad) != 0;
        }
#pragma unroll
        for (int c = 0; c < NC; ++c)
#pragma unroll
            for (int e = 0; e < E; ++e) acc[c][e] = f32x4{0.f, 0.f, 0.f, 0.f};
        if (!odd) {
#pragma unroll
            for (int st = 0; st < 16; ++st)
#pragma unroll
                for (int c = 0; c < NC; ++c)
#pragma unroll
                    for (int e = 0; e < E; ++e)
                        acc[c][e] =
                            __builtin_amdgcn_mfma_f32_16x16x4f32(vr[st][c][e], pf[st >> 2][st & 3], acc[c][e], 0, 0, 0);
            if (!partial) return;
            uint32_t least = ~0u;
#pragma unroll
            for (int c = 0; c < NC; ++c)
#pragma unroll
                for (int e = 0; e < E; ++e)
#pragma unroll
                    for (int r = 0; r < 4; ++r) {
                        const uint32_t magnitude = __float_as_uint(acc[c][e][r]) << 1;
                        least = magnitude < least ? magnitude : least;
                    }
            // (a column without keys in this block has no weights, and its state stays)
            if (__ballot(least == 0u && b * 64u < keys) == 0) return;
        }
#pragma unroll 1
        for (uint32_t only = 0; only < 16u; ++only) {
            // steps of which this lane's key lies before column `only`'s end
            const int own = int(__shfl(int(keys), int(only), 64)) - int(b * 64u + grp);
#pragma unroll
            for (int c = 0; c < NC; ++c) {
                f32x4 a[E];
#pragma unroll
                for (int e = 0; e < E; ++e) a[e] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int st = 0; st < 16; ++st)
#pragma unroll
                    for (int e = 0; e < E; ++e)
                        a[e] = __builtin_amdgcn_mfma_f32_16x16x4f32(4 * st < own ? vr[st][c][e] : -0.f,
                                                                    pf[st >> 2][st & 3], a[e], 0, 0, 0);
#pragma unroll
                for (int e = 0; e < E; ++e)
#pragma unroll
                    for (int r = 0; r < 4; ++r) acc[c][e][r] = col == only ? a[e][r] : acc[c][e][r];
            }
        }
    };

    f32x4 k0[U][4];
    load_k(W == 1 ? 0u : wv, k0);  // (ahead of q)
#pragma unroll
    for (int u = 0; u < U; ++u) {
        const f32x4 v = *reinterpret_cast<const f32x4*>(q + qoff + 16 * u + 4u * grp);
#pragma unroll
        for (int i = 0; i < 4; ++i) qf[u][i] = v[i];
        transpose4(qf[u]);
    }
    float m = 0.f, l = 0.f;
    if constexpr (W == 1) {
        f32x4 o[NC][E];
#pragma unroll
        for (int c = 0; c < NC; ++c)
#pragma unroll
            for (int e = 0; e < E; ++e) o[c][e] = f32x4{0.f, 0.f, 0.f, 0.f};
        for (uint32_t b = 0; b < nblocks; ++b) {
            f32x4 s[4], acc[NC][E];
            float vr[16][NC][E];
            const float bmax = score(b, k0, s);
            load_v(b, vr);
            const bool active = b * 64u < keys;  // a column without keys in this block keeps its state
            if (b == 0) m = bmax;
            const float mn = fmaxf(m, bmax), alpha = expf(m - mn);
            float bs;
            values(b, s, mn, vr, acc, bs);
            load_k(b + 1, k0);
            if (active) {
                m = mn;
                l = fmaf(l, alpha, bs);
#pragma unroll
                for (int c = 0; c < NC; ++c)
#pragma unroll
                    for (int e = 0; e < E; ++e)
#pragma unroll
                        for (int r = 0; r < 4; ++r) o[c][e][r] = fmaf(o[c][e][r], alpha, acc[c][e][r]);
            }
        }
        if (raw < total) {
#pragma unroll
            for (int c = 0; c < NC; ++c)
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    float* yr = y + qoff + 16 * E * c + E * (4u * grp + r);
#pragma unroll
                    for (int e = 0; e < E; ++e) yr[e] = o[c][e][r] / l;
                }
        }
    } else {
        constexpr int R = REGS / W > 0 ? REGS / W : 1;  // registers of o each wave combines: (c, r, e) order
        __shared__ float sm[W][16];
        __shared__ float ssum[W][16];
        __shared__ float sacc[W][REGS][64];
        float o[R];
#pragma unroll
        for (int i = 0; i < R; ++i) o[i] = 0.f;
        const uint32_t reg0 = wv * R;
        for (uint32_t b0 = 0; b0 < nblocks; b0 += W) {
            const uint32_t b = b0 + wv;
            f32x4 s[4];
            float vr[16][NC][E];
            if (b < nblocks) {
                const float bmax = score(b, k0, s);
                if (grp == 0) sm[wv][col] = bmax;
            }
            load_v(b, vr);  // (past the last block: its last row; a load under a condition would keep two sets alive)
            lds_barrier();
            float mn = 0.f, alpha[W], bm[W];
#pragma unroll
            for (int i = 0; i < W; ++i) bm[i] = sm[i][col];
            m = b0 == 0 ? bm[0] : m;
#pragma unroll
            for (int i = 0; i < W; ++i) {
                const bool active = (b0 + i) * 64u < keys;  // a column without keys in this block keeps its state
                const float nx = fmaxf(m, bm[i]), al = expf(m - nx);
                alpha[i] = active ? al : 1.f;
                m = active ? nx : m;
                if (uint32_t(i) == wv) mn = m;
            }
            if (b < nblocks) {
                f32x4 acc[NC][E];
                float bs;
                values(b, s, mn, vr, acc, bs);
                if (grp == 0) ssum[wv][col] = bs;
#pragma unroll
                for (int c = 0; c < NC; ++c)
#pragma unroll
                    for (int r = 0; r < 4; ++r)
#pragma unroll
                        for (int e = 0; e < E; ++e) sacc[wv][(c * 4 + r) * E + e][lane] = acc[c][e][r];
            }
            load_k(b + W, k0);
            lds_barrier();
            if (reg0 < uint32_t(REGS)) {
#pragma unroll
                for (int i = 0; i < W; ++i) {
                    const bool active = (b0 + i) * 64u < keys;
                    const float sum = ssum[i][col];
                    l = active ? fmaf(l, alpha[i], sum) : l;
#pragma unroll
                    for (int j = 0; j < R; ++j) {
                        const float v = sacc[i][reg0 + j][lane];
                        o[j] = active ? fmaf(o[j], alpha[i], v) : o[j];
                    }
                }
            }
            lds_barrier();
        }
        if (raw < total && reg0 < uint32_t(REGS)) {
#pragma unroll
            for (int j = 0; j < R; ++j) {
                const uint32_t id = reg0 + j, e = id % E, r = id / E % 4u, c = id / E / 4u;
                y[qoff + 16 * E * c + E * (4u * grp + r) + e] = o[j] / l;
            }
        }
    }
}

// One query row (a decode step), G = q_heads / kv_heads of 1, 2 or 4. A workgroup per KV head would use kv_heads CUs, and one
// CU draws its K and V at about 50 GB/s (8 heads, 700 keys: 36.6 us, 1500: 64.8); so the key blocks spread over the chip,
// in three launches over a workspace: the scores and the blocks' maxima; the blocks' sums and values against the running
// maximum (a prefix of those); the ordered combine. The same arithmetic as above, in the same order. 16 heads, 8 KV heads,
// 700 keys: 536 us on the vector ALUs of 16 blocks, 4.5 + 6.2 + 3.5 here.
struct RowWorkspace {
    float *s, *bmax, *m, *sum, *acc;  // [qh][64 nb], [qh][nb] three times, [qh][nb][HD]
    __host__ __device__ RowWorkspace(float* base, uint32_t qh, uint32_t nb)
        : s(base), bmax(s + size_t(qh) * nb * 64), m(bmax + size_t(qh) * nb), sum(m + size_t(qh) * nb),
          acc(sum + size_t(qh) * nb) {}
    static uint64_t bytes(uint64_t qh, uint64_t nb, uint64_t hd) { return qh * nb * (67 + hd) * 4; }
};

// block (key block b, KV head): wave w scores keys 64 b + 16 w .. + 15 for the G heads (a 16-column tile, one chain)
template <int HD, int G>
__global__ __launch_bounds__(256) void k_row_scores(const float* __restrict__ q, const float* __restrict__ kc,
                                                    RowWorkspace ws, uint32_t q_row0, uint32_t past, uint32_t qh,
                                                    uint32_t kvh, float scale) {
    constexpr int U = HD / 16;
    __shared__ float sm[4][16];
    const uint32_t lane = threadIdx.x & 63u, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t col = lane & 15u, grp = lane >> 4, b = blockIdx.x, nb = gridDim.x, kvhead = blockIdx.y;
    const uint32_t keys = past + 1u, j0 = b * 64u + 16u * wv, j = j0 + col, head = kvhead * G + col % G;
    const float* kp = kc + (size_t(j < keys ? j : keys - 1u) * kvh + kvhead) * HD + 4u * grp;
    const float* qp = q + (size_t(q_row0) * qh + head) * HD + 4u * grp;
    f32x4 kr[U], qr[U];
#pragma unroll
    for (int u = 0; u < U; ++u) kr[u] = *reinterpret_cast<const f32x4*>(kp + 16 * u);
#pragma unroll
    for (int u = 0; u < U; ++u) qr[u] = *reinterpret_cast<const f32x4*>(qp + 16 * u);
    __builtin_amdgcn_sched_barrier(0);
    float kf[U][4], qf[U][4];
#pragma unroll
    for (int u = 0; u < U; ++u) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            kf[u][i] = kr[u][i];
            qf[u][i] = qr[u][i];
        }
        transpose4(kf[u]);
        transpose4(qf[u]);
    }
    __builtin_amdgcn_sched_barrier(0);
    f32x4 s = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
        for (int i = 0; i < 4; ++i) s = __builtin_amdgcn_mfma_f32_16x16x4f32(kf[u][i], qf[u][i], s, 0, 0, 0);
    float mx = -INFINITY;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        s[r] = j0 + 4u * grp + r < keys ? s[r] * scale : -INFINITY;
        mx = fmaxf(mx, s[r]);
    }
    mx = fast::cross_rows_max(mx);
    if (lane < 16u) sm[wv][col] = mx;
    if (col < uint32_t(G)) *reinterpret_cast<f32x4*>(ws.s + size_t(head) * nb * 64 + j0 + 4u * grp) = s;
    __syncthreads();
    if (threadIdx.x < uint32_t(G))
        ws.bmax[size_t(kvhead * G + threadIdx.x) * nb + b] =
            fmaxf(fmaxf(sm[0][threadIdx.x], sm[1][threadIdx.x]), fmaxf(sm[2][threadIdx.x], sm[3][threadIdx.x]));
}

// block (key block b, KV head), one thread per head and dimension: the weights against the running maximum, their sum,
// the block's values
template <int HD, int G>
__global__ __launch_bounds__(HD* G < 64 ? 64 : HD * G) void k_row_values(const float* __restrict__ vc, RowWorkspace ws,
                                                                         uint32_t past, uint32_t kvh) {
    constexpr int NT = HD * G < 64 ? 64 : HD * G;
    __shared__ __align__(16) float ps[G][64];
    const uint32_t t = threadIdx.x, b = blockIdx.x, nb = gridDim.x, kvhead = blockIdx.y;
    const uint32_t h = t / HD, d = t % HD, keys = past + 1u;
    const uint32_t count = keys - b * 64u < 64u ? keys - b * 64u : 64u;
    const float* vp = vc + (size_t(b) * 64u * kvh + kvhead) * HD;
    float v[64];
#pragma unroll
    for (uint32_t j = 0; j < 64; ++j) v[j] = vp[size_t((j < count ? j : count - 1u) * kvh * HD) + d];
    __builtin_amdgcn_sched_barrier(0);
    if (t < 64u) {  // one wave: the running maxima, then the weights of key `t`
#pragma unroll
        for (int g = 0; g < G; ++g) {
            const uint32_t head = kvhead * G + g;
            const float score = ws.s[size_t(head) * nb * 64 + b * 64u + t];
            float mx = ws.bmax[size_t(head) * nb];
            for (uint32_t i = t; i <= b; i += 64u) mx = fmaxf(mx, ws.bmax[size_t(head) * nb + i]);
            mx = fast::wave_max(mx);
            ps[g][t] = expf(score - mx);
            if (t == 0) ws.m[size_t(head) * nb + b] = mx;
        }
    }
    lds_barrier();
    if (h >= uint32_t(G)) return;
    float acc = 0.f, sum = 0.f;
    if (count == 64u) {
#pragma unroll
        for (int j = 0; j < 64; j += 4) {
            const f32x4 w = *reinterpret_cast<const f32x4*>(&ps[h][j]);
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                sum += w[e];
                acc = fmaf(w[e], v[j + e], acc);
            }
        }
    } else {
#pragma unroll
        for (uint32_t j = 0; j < 64; ++j)
            if (j < count) {
                const float w = ps[h][j];
                sum += w;
                acc = fmaf(w, v[j], acc);
            }
    }
    const size_t at = size_t(kvhead * G + h) * nb + b;
    ws.acc[at * HD + d] = acc;
    if (d == 0) ws.sum[at] = sum;
}

// block (query head), one thread per dimension: the blocks in order, 64 at a time
template <int HD>
__global__ __launch_bounds__(HD < 64 ? 64 : HD) void k_row_combine(RowWorkspace ws, float* __restrict__ y, uint32_t q_row0,
                                                                   uint32_t qh, uint32_t nb) {
    __shared__ float al[64], bs[64];
    const uint32_t t = threadIdx.x, head = blockIdx.x, d = t % HD;
    const float* acc = ws.acc + size_t(head) * nb * HD + d;
    const float* m = ws.m + size_t(head) * nb;
    float l = 0.f, o = 0.f;
    for (uint32_t b0 = 0; b0 < nb; b0 += 64u) {
        if (t < 64u) {
            const uint32_t b = b0 + t < nb ? b0 + t : nb - 1u;
            const float before = b == 0 ? ws.bmax[size_t(head) * nb] : m[b - 1u];
            al[t] = expf(before - m[b]);
            bs[t] = ws.sum[size_t(head) * nb + b];
        }
        __syncthreads();
        const uint32_t n = nb - b0 < 64u ? nb - b0 : 64u;
#pragma unroll 8
        for (uint32_t i = 0; i < n; ++i) {
            l = fmaf(l, al[i], bs[i]);
            o = fmaf(o, al[i], acc[size_t(b0 + i) * HD]);
        }
        __syncthreads();
    }
    if (t < uint32_t(HD)) y[(size_t(q_row0) * qh + head) * HD + d] = o / l;
}

template <int HD>
static bool launch_attention(const float* q, const float* kc, const float* vc, float* y, uint32_t rows, uint32_t q_row0,
                             uint32_t past, uint32_t qh, uint32_t kvh, float scale, void* workspace,
                             hipStream_t s) {
    const uint64_t tiles = (uint64_t(rows) * (qh / kvh) + 15) / 16;
    const uint32_t group = qh / kvh, nb = past / 64u + 1u;
    // (three launches against one: at 64 and 128 dimensions they win from the first key, 63 keys 10 us against 14; below,
    // where a block is little work, from eight blocks on)
    const bool spread = workspace && rows == 1 && (HD >= 64 || nb >= 8) && (group == 1 || group == 2 || group == 4) &&
                        uint64_t(64) * kvh * HD < (1ull << 30) && RowWorkspace::bytes(qh, nb, HD) <= kWorkspaceBytes;
    // Of a few keys a tile's loads and exchanges of 64 are most of its time, and the general kernel, a workgroup per row and
    // head, is done before. 16 heads, general kernel against this file's, us: 1 key of 16 dimensions 3.2 / 5.2, 9 keys 4.9 / 5.3,
    // 12 keys 5.5 / 5.3; 1 row at 9 keys of 64, over the chip, 7.7 / 9.4, at 16 9.5 / 9.6; 9 rows of 128 12.7 / 14.8, 12 rows
    // 14.1 / 14.8, 16 rows 15.3 / 14.9; but 1 row at 8 keys of 128, over the chip, 12.2 / 10.1. Many rows and heads take longer
    // than a tile each on its CU (512 heads, 8 rows of 16: 6.6 / 5.7), but not than the tiles' second turn (9 rows of 128: 17.9
    // / 29.6).
    const uint32_t few = HD == 64 && spread ? 13 : HD == 128 ? (spread ? 0 : 12) : 10;
    const bool second = HD >= 32 && tiles * kvh > 256 && tiles * kvh <= 384;
    if (uint64_t(past) + rows <= few && (uint64_t(rows) * qh <= 3072 || second)) return false;
    if (spread) {
        const RowWorkspace ws(static_cast<float*>(workspace), qh, nb);
        auto go = [&](auto scores, auto values, uint32_t threads) {
            hipLaunchKernelGGL(scores, dim3(nb, kvh), dim3(256), 0, s, q, kc, ws, q_row0, past, qh, kvh, scale);
            hipLaunchKernelGGL(values, dim3(nb, kvh), dim3(threads < 64 ? 64 : threads), 0, s, vc, ws, past, kvh);
        };
        if (group == 1) go(k_row_scores<HD, 1>, k_row_values<HD, 1>, HD);
        if (group == 2) go(k_row_scores<HD, 2>, k_row_values<HD, 2>, 2 * HD);
        if (group == 4) go(k_row_scores<HD, 4>, k_row_values<HD, 4>, 4 * HD);
        hipLaunchKernelGGL(k_row_combine<HD>, dim3(qh), dim3(HD < 64 ? 64 : HD), 0, s, ws, y, q_row0, qh, nb);
        return true;
    }
    // One wave per tile once the tiles alone give each of the chip's 1024 SIMDs one, else eight waves share a tile. 16 heads,
    // 8 KV heads, one against eight waves: 512 rows (512 tiles) 60.1 / 54.1 us, 512 after 2048 272 / 224, 1024 113 / 148,
    // 1536 168 / 264, 2048 243 / 433, 4096 918 / 1520. (With the tiles of one KV head before the next one's, the last head's
    // longest began when the others' shortest ended: 1536 rows 284 us, 2048 447, slower than eight waves, 4096 1324.)
    if (tiles * kvh >= 1024)
        hipLaunchKernelGGL((k_attention_mfma<HD, 1>), dim3(uint32_t((tiles + 3) / 4) * kvh), dim3(256), 0, s, q, kc, vc, y,
                           rows, q_row0, past, qh, kvh, scale);
    else
        hipLaunchKernelGGL((k_attention_mfma<HD, 8>), dim3(uint32_t(tiles), kvh), dim3(512), 0, s, q, kc, vc, y, rows,
                           q_row0, past, qh, kvh, scale);
    return true;
}

bool attention(const float* q, const float* kc, const float* vc, float* y, uint32_t rows, uint32_t q_row0, uint32_t past,
               uint32_t qh, uint32_t kvh, uint32_t hd, float scale, void* workspace, hipStream_t s) {
    if (!aligned16(q) || !aligned16(kc) || !aligned16(vc) || uint64_t(rows) * (qh / kvh) > 0x7FFFFFFFull) return false;
    switch (hd) {
        case 16: return launch_attention<16>(q, kc, vc, y, rows, q_row0, past, qh, kvh, scale, workspace, s);
        case 32: return launch_attention<32>(q, kc, vc, y, rows, q_row0, past, qh, kvh, scale, workspace, s);
        case 64: return launch_attention<64>(q, kc, vc, y, rows, q_row0, past, qh, kvh, scale, workspace, s);
        case 128: return launch_attention<128>(q, kc, vc, y, rows, q_row0, past, qh, kvh, scale, workspace, s);
        default: return false;
    }
}

}  // namespace f32k
}  // namespace lrm
