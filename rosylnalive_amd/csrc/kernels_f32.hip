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
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));

// ---------------------------------------------------------------- matmul_bf16w
// The operand of step s of a 16x16x4 MFMA holds k = 4 s + g in lane group g = lane / 16. A staged tile therefore keeps
// each row's k values by group, [row][g][k / 4], so that one LDS read gives a lane four (x, 16 bytes) or four (w, 8
// bytes) consecutive steps. Row strides 68 and 36 words: the 16 rows of a group start in distinct banks.
constexpr int KS = 64;            // k per staged tile
constexpr int XROW = KS + 4;      // words per staged x row
constexpr int WROW = KS / 2 + 4;  // words per staged w row (bf16 pairs)

// k at or past the end: x = +0 and w = -0, whose product -0 leaves every chain value as it is, -0 included.
constexpr uint32_t kNegZeroPair = 0x80008000u;

// One block computes a (16 WR TM) x (16 WC TN) tile with WR x WC waves of TM x TN MFMA tiles. D register sets of the
// next tiles are in flight while the current one multiplies (a step of 64 k takes 0.3 us at one tile per wave, a load
// from HBM 1-2 us), two LDS stages, one LDS-only barrier per step. The loop runs whole groups of D steps; steps past k
// multiply the padding.
// VEC: x and w 16-byte aligned, k a multiple of 8; otherwise element loads.
template <int WR, int WC, int TM, int TN, int D, bool VEC>
__global__ __launch_bounds__(256) void k_matmul_mfma(const float* __restrict__ x, const uint16_t* __restrict__ w,
                                                     float* __restrict__ y, uint32_t m, uint32_t n, uint32_t k) {
    static_assert(WR * WC == 4, "four waves");
    constexpr int BM = 16 * WR * TM, BN = 16 * WC * TN;
    constexpr int XQ = BM * (KS / 4) / 256, WQ = BN * (KS / 8) / 256;  // 16-byte chunks per thread
    static_assert(XQ >= 1 && WQ >= 1, "whole chunks");
    __shared__ float xs[2][BM * XROW];
    __shared__ uint32_t ws[2][BN * WROW];
    const uint32_t t = threadIdx.x, lane = t & 63u, wv = t >> 6, wr = wv / WC, wc = wv % WC;
    const uint32_t i0 = blockIdx.y * BM, j0 = blockIdx.x * BN;
    // chunk q of this thread: x row xr(q), k 4 xc ..; a wave's four rows are 4 apart (distinct banks when stored)
    const uint32_t xc = t & 15u, xr0 = ((t >> 4) & 3u) * 4u + (t >> 6);
    const uint32_t wcx = t & 7u, wr0 = t >> 3;
    u32x4 xreg[D][XQ], wreg[D][WQ];

    auto load = [&](int d, uint32_t k0) {
#pragma unroll
        for (int q = 0; q < XQ; ++q) {
            uint32_t row = i0 + xr0 + 16u * q;
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
            uint32_t col = j0 + wr0 + 32u * q;
            col = col < n ? col : n - 1u;
            const uint32_t kk = k0 + 8u * wcx;
            if constexpr (VEC) {
                wreg[d][q] = *reinterpret_cast<const u32x4*>(w + size_t(col) * k + (kk < k ? kk : 0u));
            } else {
#pragma unroll
                for (uint32_t e = 0; e < 4; ++e) {
                    const uint32_t a = kk + 2u * e, b = a + 1u;
                    const uint32_t lo = w[size_t(col) * k + (a < k ? a : 0u)], hi = w[size_t(col) * k + (b < k ? b : 0u)];
                    wreg[d][q][e] = (a < k ? lo : 0x8000u) | (b < k ? hi << 16 : 0x80000000u);
                }
            }
        }
    };
    auto store = [&](int d, int buf, uint32_t k0) {
#pragma unroll
        for (int q = 0; q < XQ; ++q) {
            const uint32_t kk = k0 + 4u * xc;
            float* p = &xs[buf][(xr0 + 16u * q) * XROW + xc];
#pragma unroll
            for (uint32_t g = 0; g < 4; ++g) {
                const bool in = VEC ? kk < k : kk + g < k;
                p[g * (KS / 4)] = in ? __uint_as_float(xreg[d][q][g]) : 0.f;
            }
        }
#pragma unroll
        for (int q = 0; q < WQ; ++q) {
            u32x4 v = wreg[d][q];
            if (VEC && k0 + 8u * wcx >= k) v = u32x4{kNegZeroPair, kNegZeroPair, kNegZeroPair, kNegZeroPair};
            uint32_t* p = &ws[buf][(wr0 + 32u * q) * WROW + wcx];
            p[0] = (v[0] & 0xFFFFu) | (v[2] << 16);
            p[8] = (v[0] >> 16) | (v[2] & 0xFFFF0000u);
            p[16] = (v[1] & 0xFFFFu) | (v[3] << 16);
            p[24] = (v[1] >> 16) | (v[3] & 0xFFFF0000u);
        }
    };

    f32x4 acc[TM][TN];
#pragma unroll
    for (int a = 0; a < TM; ++a)
#pragma unroll
        for (int b = 0; b < TN; ++b) acc[a][b] = f32x4{0.f, 0.f, 0.f, 0.f};
    const uint32_t r16 = lane & 15u, grp = lane >> 4;
    auto compute = [&](int buf) {
        const float* xb = &xs[buf][(wr * TM * 16u + r16) * XROW + grp * (KS / 4)];
        const uint32_t* wb = &ws[buf][(wc * TN * 16u + r16) * WROW + grp * (KS / 8)];
#pragma unroll
        for (int q = 0; q < KS / 16; ++q) {
            f32x4 av[TM];
            u32x2 bv[TN];
#pragma unroll
            for (int a = 0; a < TM; ++a) av[a] = *reinterpret_cast<const f32x4*>(xb + a * 16 * XROW + 4 * q);
#pragma unroll
            for (int b = 0; b < TN; ++b) bv[b] = *reinterpret_cast<const u32x2*>(wb + b * 16 * WROW + 2 * q);
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int a = 0; a < TM; ++a)
#pragma unroll
                    for (int b = 0; b < TN; ++b) {
                        const uint32_t h = bv[b][i >> 1];
                        acc[a][b] = __builtin_amdgcn_mfma_f32_16x16x4f32(
                            av[a][i], __uint_as_float((i & 1) ? h & 0xFFFF0000u : h << 16), acc[a][b], 0, 0, 0);
                    }
        }
    };

#pragma unroll
    for (int d = 0; d < D; ++d) load(d, uint32_t(d) * KS);
    store(0, 0, 0);
    lds_barrier();
    for (uint32_t k0 = 0; k0 < k; k0 += D * KS) {
#pragma unroll
        for (int d = 0; d < D; ++d) {
            load(d, k0 + uint32_t(d + D) * KS);  // this set's tile is in LDS
            compute(d & 1);
            store((d + 1) % D, (d + 1) & 1, k0 + uint32_t(d + 1) * KS);
            lds_barrier();
        }
    }
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

// One or two rows of x (a decode step): an output is one dependent chain, so its k fused adds bound the kernel (5-6
// cycles each: the add and its share of the LDS reads), not the weights. A block owns 32 columns: wave 4 runs the chains
// (lane = column + 32 row), waves 0-3 load the weights (16 bytes per lane, D tiles of 128 k in flight), widen them to
// float32 into LDS, two stages, one barrier per tile. 32 columns and not 64: the weights of one block come through one
// CU, and at 64 columns that stream is slower than the chain.
constexpr int ROW_C = 32, ROW_KT = 128, ROW_STRIDE = ROW_KT + 4, ROW_D = 4;
__global__ __launch_bounds__(320) void k_matmul_row(const float* __restrict__ x, const uint16_t* __restrict__ w,
                                                    float* __restrict__ y, uint32_t m, uint32_t n, uint32_t k) {
    __shared__ float ws[2][ROW_C * ROW_STRIDE];
    __shared__ float xs[2][2][ROW_KT];
    const uint32_t t = threadIdx.x, j0 = blockIdx.x * ROW_C;
    const uint32_t tiles = (k + ROW_KT - 1) / ROW_KT, rounds = (tiles + ROW_D - 1) / ROW_D;
    if (t < 256) {
        const uint32_t c = t & 15u, col0 = t >> 4;  // chunk: 8 k of column col0 (and col0 + 16)
        const uint32_t xrow = (t >> 5) < m ? t >> 5 : m - 1u, xc = t & 31u;
        u32x4 wreg[ROW_D][2];
        f32x4 xreg[ROW_D];
        auto load = [&](int d, uint32_t k0) {
#pragma unroll
            for (int q = 0; q < 2; ++q) {
                uint32_t col = j0 + col0 + 16u * q;
                col = col < n ? col : n - 1u;
                const uint32_t kk = k0 + 8u * c;
                wreg[d][q] = *reinterpret_cast<const u32x4*>(w + size_t(col) * k + (kk < k ? kk : 0u));
            }
            if (t < 64) {
                const uint32_t kk = k0 + 4u * xc;
                xreg[d] = *reinterpret_cast<const f32x4*>(x + size_t(xrow) * k + (kk < k ? kk : 0u));
            }
        };
        auto store = [&](int d, int buf, uint32_t k0) {
            const bool in = k0 + 8u * c < k;
#pragma unroll
            for (int q = 0; q < 2; ++q) {
                u32x4 v = wreg[d][q];
                if (!in) v = u32x4{kNegZeroPair, kNegZeroPair, kNegZeroPair, kNegZeroPair};
                float* p = &ws[buf][(col0 + 16u * q) * ROW_STRIDE + 8u * c];
                f32x4 a, b;
#pragma unroll
                for (int e = 0; e < 2; ++e) {
                    a[2 * e] = __uint_as_float(v[e] << 16);
                    a[2 * e + 1] = __uint_as_float(v[e] & 0xFFFF0000u);
                    b[2 * e] = __uint_as_float(v[e + 2] << 16);
                    b[2 * e + 1] = __uint_as_float(v[e + 2] & 0xFFFF0000u);
                }
                *reinterpret_cast<f32x4*>(p) = a;
                *reinterpret_cast<f32x4*>(p + 4) = b;
            }
            if (t < 64) {
                f32x4 v = xreg[d];
                if (k0 + 4u * xc >= k) v = f32x4{0.f, 0.f, 0.f, 0.f};
                *reinterpret_cast<f32x4*>(&xs[buf][t >> 5][4u * xc]) = v;
            }
        };
#pragma unroll
        for (int d = 0; d < ROW_D; ++d) load(d, uint32_t(d) * ROW_KT);
        store(0, 0, 0);
        lds_barrier();
        for (uint32_t r = 0; r < rounds; ++r) {
            const uint32_t k0 = r * ROW_D * ROW_KT;
#pragma unroll
            for (int d = 0; d < ROW_D; ++d) {
                load(d, k0 + uint32_t(d + ROW_D) * ROW_KT);
                store((d + 1) % ROW_D, (d + 1) & 1, k0 + uint32_t(d + 1) * ROW_KT);
                lds_barrier();
            }
        }
    } else {
        const uint32_t lane = t - 256u, col = lane & 31u, row = lane >> 5;
        float acc = 0.f;
        lds_barrier();
        for (uint32_t r = 0; r < rounds; ++r) {
#pragma unroll
            for (int d = 0; d < ROW_D; ++d) {
                const float* wp = &ws[d & 1][col * ROW_STRIDE];
                const float* xp = xs[d & 1][row];
#pragma unroll
                for (int q = 0; q < ROW_KT / 4; ++q) {
                    const f32x4 a = *reinterpret_cast<const f32x4*>(xp + 4 * q);
                    const f32x4 b = *reinterpret_cast<const f32x4*>(wp + 4 * q);
#pragma unroll
                    for (int e = 0; e < 4; ++e) acc = fmaf(a[e], b[e], acc);
                }
                lds_barrier();
            }
        }
        if (row < m && j0 + col < n) y[size_t(row) * n + j0 + col] = acc;
    }
}

static bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }

template <int WR, int WC, int TM, int TN, int D>
static void launch_mfma(bool vec, const float* x, const uint16_t* w, float* y, uint32_t m, uint32_t n, uint32_t k,
                        hipStream_t s) {
    constexpr uint32_t BM = 16 * WR * TM, BN = 16 * WC * TN;
    const dim3 grid((n + BN - 1) / BN, (m + BM - 1) / BM);
    if (vec)
        hipLaunchKernelGGL((k_matmul_mfma<WR, WC, TM, TN, D, true>), grid, dim3(256), 0, s, x, w, y, m, n, k);
    else
        hipLaunchKernelGGL((k_matmul_mfma<WR, WC, TM, TN, D, false>), grid, dim3(256), 0, s, x, w, y, m, n, k);
}

void matmul_bf16w(const float* x, const uint16_t* w, float* y, uint32_t m, uint32_t n, uint32_t k, hipStream_t s) {
    const bool vec = k % 8 == 0 && aligned16(x) && aligned16(w);
    if (m <= 2 && vec) {
        hipLaunchKernelGGL(k_matmul_row, dim3((n + ROW_C - 1) / ROW_C), dim3(320), 0, s, x, w, y, m, n, k);
        return;
    }
    // 64 x 64 tiles when they give every CU two blocks, else 32 x 32 (four times the blocks), or 16 x 64 for the rows
    // of one MFMA tile
    const uint64_t big = uint64_t((m + 63) / 64) * ((n + 63) / 64);
    if (m <= 16)
        launch_mfma<1, 4, 1, 1, 4>(vec, x, w, y, m, n, k, s);
    else if (big >= 512)
        launch_mfma<2, 2, 2, 2, 2>(vec, x, w, y, m, n, k, s);
    else
        launch_mfma<2, 2, 1, 1, 4>(vec, x, w, y, m, n, k, s);
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

__device__ __forceinline__ bool finite(float v) { return (__float_as_uint(v) & 0x7F800000u) != 0x7F800000u; }

template <int HD, int W>
__global__ __launch_bounds__(W == 1 ? 256 : 64 * W) void k_attention_mfma(
    const float* __restrict__ q, const float* __restrict__ kc, const float* __restrict__ vc, float* __restrict__ y,
    uint32_t rows, uint32_t q_row0, uint32_t past, uint32_t qh, uint32_t kvh, float scale) {
    constexpr int E = HD % 64 == 0 ? 4 : 1, NC = HD / (16 * E), U = HD / 16;
    constexpr int REGS = HD / 4;  // O registers per lane: 16 columns x HD over 64 lanes
    const uint32_t lane = threadIdx.x & 63u, wv = threadIdx.x >> 6, col = lane & 15u, grp = lane >> 4;
    const uint32_t group = qh / kvh, kvhead = blockIdx.y, total = rows * group, tiles = (total + 15u) / 16u;
    const uint32_t tb = W == 1 ? blockIdx.x * 4u + wv : blockIdx.x;
    if (tb >= tiles) return;
    const uint32_t tile = tiles - 1u - tb;  // the longest first
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
#pragma unroll
    for (int u = 0; u < U; ++u) {
        const f32x4 v = *reinterpret_cast<const f32x4*>(q + qoff + 16 * u + 4u * grp);
#pragma unroll
        for (int i = 0; i < 4; ++i) qf[u][i] = v[i];
        transpose4(qf[u]);
    }

    // scores of block b: s[t][r] = key 64 b + 16 t + 4 grp + r (times scale); returns the block's maximum over this
    // column's keys (-inf for none)
    auto score = [&](uint32_t b, f32x4 (&s)[4]) {
        float mx = -INFINITY;
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            const uint32_t j = b * 64u + 16u * t + col;
            const float* kr = kb + size_t(j < max_keys ? j : max_keys - 1u) * kv_stride;
            f32x4 a = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const f32x4 kv = *reinterpret_cast<const f32x4*>(kr + 16 * u);
                float kf[4] = {kv[0], kv[1], kv[2], kv[3]};
                transpose4(kf);
#pragma unroll
                for (int i = 0; i < 4; ++i) a = __builtin_amdgcn_mfma_f32_16x16x4f32(kf[i], qf[u][i], a, 0, 0, 0);
            }
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                // a key past the column's own scores -inf: weight 0 (or NaN where every score is -inf or NaN, and the
                // reference's weights are NaN too)
                s[t][r] = b * 64u + 16u * t + 4u * grp + r < keys ? a[r] * scale : -INFINITY;
                mx = fmaxf(mx, s[t][r]);
            }
        }
        return fast::cross_rows_max(mx);
    };

    // the block's values and sum against the maximum mn: acc (register (c, e, r) = dimension 16 E c + E (4 grp + r) + e
    // of this column), bs the sum of the weights
    auto values = [&](uint32_t b, const f32x4 (&s)[4], float mn, f32x4 (&acc)[NC][E], float& bs) {
        float pf[4][4];
#pragma unroll
        for (int t = 0; t < 4; ++t) {
#pragma unroll
            for (int r = 0; r < 4; ++r)
                pf[t][r] = expf(s[t][r] - mn);
            transpose4(pf[t]);
        }
        f32x4 sum = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int st = 0; st < 16; ++st) sum = __builtin_amdgcn_mfma_f32_16x16x4f32(1.f, pf[st >> 2][st & 3], sum, 0, 0, 0);
        bs = sum[0];
        // this lane's E values of tile group c at step st (a key past the tile's last: its last)
        auto value = [&](int st, int c, float (&vv)[E]) {
            const uint32_t j = b * 64u + 4u * st + grp;
            const float* vr = vb + size_t(j < max_keys ? j : max_keys - 1u) * kv_stride + 16 * E * c;
            if constexpr (E == 4) {
                const f32x4 l = *reinterpret_cast<const f32x4*>(vr);
#pragma unroll
                for (int e = 0; e < 4; ++e) vv[e] = l[e];
            } else {
                vv[0] = vr[0];
            }
        };
        // A key past a column's own has weight 0, which leaves the chain as it is only while its value is finite: where
        // a block with such keys holds an infinity or a NaN, each column runs alone with those values zeroed.
        bool odd = false;
        if (b * 64u + 64u > first_keys) {
            uint32_t bad = 0;
#pragma unroll 4
            for (int st = 0; st < 16; ++st)
#pragma unroll
                for (int c = 0; c < NC; ++c) {
                    float vv[E];
                    value(st, c, vv);
#pragma unroll
                    for (int e = 0; e < E; ++e) bad |= uint32_t(!finite(vv[e]));
                }
            odd = __ballot(bad != 0u) != 0;
        }
#pragma unroll
        for (int c = 0; c < NC; ++c)
#pragma unroll
            for (int e = 0; e < E; ++e) acc[c][e] = f32x4{0.f, 0.f, 0.f, 0.f};
        if (!odd) {
#pragma unroll
            for (int st = 0; st < 16; ++st)
#pragma unroll
                for (int c = 0; c < NC; ++c) {
                    float vv[E];
                    value(st, c, vv);
#pragma unroll
                    for (int e = 0; e < E; ++e)
                        acc[c][e] = __builtin_amdgcn_mfma_f32_16x16x4f32(vv[e], pf[st >> 2][st & 3], acc[c][e], 0, 0, 0);
                }
            return;
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
                for (int st = 0; st < 16; ++st) {
                    float vv[E];
                    value(st, c, vv);
#pragma unroll
                    for (int e = 0; e < E; ++e)
                        a[e] = __builtin_amdgcn_mfma_f32_16x16x4f32(4 * st < own ? vv[e] : 0.f, pf[st >> 2][st & 3], a[e], 0,
                                                                    0, 0);
                }
#pragma unroll
                for (int e = 0; e < E; ++e)
#pragma unroll
                    for (int r = 0; r < 4; ++r) acc[c][e][r] = col == only ? a[e][r] : acc[c][e][r];
            }
        }
    };

    float m = 0.f, l = 0.f;
    if constexpr (W == 1) {
        f32x4 o[NC][E];
#pragma unroll
        for (int c = 0; c < NC; ++c)
#pragma unroll
            for (int e = 0; e < E; ++e) o[c][e] = f32x4{0.f, 0.f, 0.f, 0.f};
        for (uint32_t b = 0; b < nblocks; ++b) {
            f32x4 s[4], acc[NC][E];
            const float bmax = score(b, s);
            const bool active = b * 64u < keys;  // a column without keys in this block keeps its state
            if (b == 0) m = bmax;
            const float mn = fmaxf(m, bmax), alpha = expf(m - mn);
            float bs;
            values(b, s, mn, acc, bs);
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
            if (b < nblocks) {
                const float bmax = score(b, s);
                if (grp == 0) sm[wv][col] = bmax;
            }
            lds_barrier();
            float mn = 0.f, alpha[W];
#pragma unroll
            for (int i = 0; i < W; ++i) {
                alpha[i] = 1.f;
                if ((b0 + i) * 64u < keys) {
                    const float bm = sm[i][col];
                    if (b0 + i == 0) m = bm;
                    const float nx = fmaxf(m, bm);
                    alpha[i] = expf(m - nx);
                    m = nx;
                }
                if (uint32_t(i) == wv) mn = m;
            }
            if (b < nblocks) {
                f32x4 acc[NC][E];
                float bs;
                values(b, s, mn, acc, bs);
                if (grp == 0) ssum[wv][col] = bs;
#pragma unroll
                for (int c = 0; c < NC; ++c)
#pragma unroll
                    for (int r = 0; r < 4; ++r)
#pragma unroll
                        for (int e = 0; e < E; ++e) sacc[wv][(c * 4 + r) * E + e][lane] = acc[c][e][r];
            }
            lds_barrier();
#pragma unroll
            for (int i = 0; i < W; ++i)
                if ((b0 + i) * 64u < keys) {
                    l = fmaf(l, alpha[i], ssum[i][col]);
                    if (reg0 < uint32_t(REGS)) {
#pragma unroll
                        for (int j = 0; j < R; ++j) o[j] = fmaf(o[j], alpha[i], sacc[i][reg0 + j][lane]);
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

template <int HD>
static void launch_attention(const float* q, const float* kc, const float* vc, float* y, uint32_t rows, uint32_t q_row0,
                             uint32_t past, uint32_t qh, uint32_t kvh, float scale, hipStream_t s) {
    const uint64_t tiles = (uint64_t(rows) * (qh / kvh) + 15) / 16;
    // one wave per tile once the tiles alone fill the chip's 1024 SIMDs several times over; else eight waves share one
    if (tiles * kvh >= 4096)
        hipLaunchKernelGGL((k_attention_mfma<HD, 1>), dim3(uint32_t((tiles + 3) / 4), kvh), dim3(256), 0, s, q, kc, vc, y,
                           rows, q_row0, past, qh, kvh, scale);
    else
        hipLaunchKernelGGL((k_attention_mfma<HD, 8>), dim3(uint32_t(tiles), kvh), dim3(512), 0, s, q, kc, vc, y, rows,
                           q_row0, past, qh, kvh, scale);
}

bool attention(const float* q, const float* kc, const float* vc, float* y, uint32_t rows, uint32_t q_row0, uint32_t past,
               uint32_t qh, uint32_t kvh, uint32_t hd, float scale, hipStream_t s) {
    if (!aligned16(q) || !aligned16(kc) || !aligned16(vc) || uint64_t(rows) * (qh / kvh) > 0x7FFFFFFFull) return false;
    switch (hd) {
        case 16: launch_attention<16>(q, kc, vc, y, rows, q_row0, past, qh, kvh, scale, s); return true;
        case 32: launch_attention<32>(q, kc, vc, y, rows, q_row0, past, qh, kvh, scale, s); return true;
        case 64: launch_attention<64>(q, kc, vc, y, rows, q_row0, past, qh, kvh, scale, s); return true;
        case 128: launch_attention<128>(q, kc, vc, y, rows, q_row0, past, qh, kvh, scale, s); return true;
        default: return false;
    }
}

}  // namespace f32k
}  // namespace lrm
