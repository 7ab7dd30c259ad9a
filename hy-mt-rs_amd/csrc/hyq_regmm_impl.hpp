// Batched products of few tokens with the weights dequantized straight into
// MFMA operands (Weight::matmul at batch 2 .. 64, src/quant.rs:
// 272-344, on the f16-MFMA path): no LDS copy of either operand, no barrier
// in the K loop.
//
// Bound. A few tokens leave the matrix cores little to do: the product costs
// the weights' stream from HBM and each CU's load path - a wave's weight
// load touches 32 rows' cache lines, and its token fragments (4 KiB per 64
// columns and 32 tokens) come from L2 for every 32 rows. Timing-only variants
// at Q4_K [14336 x 4096], 21 tokens (24.9 us with 8 waves): weights read as
// contiguous KiBs 20.5, no token loads 20.5, both 17.8, no dequantization
// 23.9. A 128-token tile of the LDS engine (hyq_tile.hpp) spends the same
// MFMAs on 21 tokens as on 128 and meets a barrier every 64 columns.
// Measured, with the f16 rows' launch (LDS engine -> this): Q2_0C
// [6144 x 2048] 21 tokens 17.0 -> 10.1 us, 64 tokens 22.4 -> 12.1; Q4_K
// [14336 x 4096] 21 tokens 44.5 -> 23.4, 64 tokens 48.5 -> 28.4; Q6_K
// [4096 x 4096] 20 tokens 14.2 (where it stays with the engine: hyq_regmm.hip).
//
// Form. A workgroup owns 32 weight rows against the TB blocks of 32 tokens; its
// waves split K in 64-column steps, each wave with all of the workgroup's rows
// and tokens, and meet once, in LDS, where the waves' sums are added in wave
// order. Lane l of a wave is weight row l % 32 and
// half h = l / 32 of a step's columns (Deq<F>'s halves): the 32 values it
// dequantizes are four A fragments of v_mfma_f32_32x32x16_f16 as they are -
// a 16-deep step may take its columns in any order as long as both operands
// take the same - so the token fragments, kept in fragment order (8
// consecutive columns of a token per 16-byte piece), are read at the pieces
// of those columns. The packed bytes of the next 256 columns are in registers
// while 256 are multiplied.
//
// GU is the gate/up product of a gated FFN: the tile's rows are 16 of gate and
// the same 16 of up in turns of two, so that a thread's four rows of the final
// sum are two of each and it writes silu(g) * u. The MoE's shared experts at
// 64 tokens (Q8_0, 2 x [1536 x 2048], then [2048 x 1536]): 15.9 and 12.7 us in
// the LDS engine, whose grids are 48 and 32 workgroups, 11.2 and 10.8 here; the
// layer 151.6 -> 144.7 us, at 6 tokens 98.2 -> 89.9.
//
// Every weight is the same f16 value as in the LDS engine (one fma
// bit-identical to the decoder, one rounding); an output's terms are summed
// in another order. A token's result depends on its own row and the weight's
// shape only: the same bits at any batch that runs this form.
#pragma once

#include <hip/hip_runtime.h>

#include "hyq_tile.hpp"

#pragma clang fp contract(off)

namespace hyq {
namespace regmm {

using namespace tile;

// The 8-column piece (of the 64-column step's eight) that fragment i of half
// h holds: piece g of a block of c tokens is at 8 c g halves of the step's
// fragment-order run.
template <int F> __device__ constexpr int piece(int i, int h)
{
    return (i < 2 ? Deq<F>::c0(h) + 8 * i : Deq<F>::c1(h) + 8 * (i - 2)) / 8;
}

// Waves of a workgroup. Four, so that a CU holds up to four workgroups at the
// 128 registers of a wave and one's loads run under another's products; with
// 8 and 16 waves Q4_K [14336 x 4096] at 21 tokens took 24.9 and 28.7 us
// against 23.4.
constexpr int WAVES = 4;

// Waves per SIMD: what two 256-column blocks of packed bytes leave room for.
template <int F, int TB> constexpr int occupancy()
{
    return F == Q6_K || (TB > 1 && (F == Q4_K || F == Q8_0)) ? 3 : 4;
}

struct Args {
    WView w, up; // up: GU, w is gate
    float *y;
    const float *residual;
    int rows, rtiles, K, N, kslices; // rtiles: of 32 rows (GU: 16 of each)
    const _Float16 *xh;              // fragment order
    const float *rscale;
    float *part; // [kslices][N][rows] when kslices > 1
};

template <int F, int TB, bool GU>
__global__ __launch_bounds__(64 * WAVES, (occupancy<F, TB>())) void regmm_kernel(Args a)
{
    using D = Deq<F>;
    __shared__ float4 red[TB][WAVES][4][64];
    const int per = (a.rtiles + 7) / 8;
    const int T = (int)(blockIdx.x % 8) * per + (int)(blockIdx.x / 8); // XCD-contiguous
    if (T >= a.rtiles) return;
    const int M = a.rows, K = a.K, N = a.N;
    const int m0 = T * (GU ? 16 : 32);
    const int t = threadIdx.x, lane = t & 63, h = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane(t >> 6);

    // this wave's steps, whole 256-column blocks of four (Q8_0's last may be less)
    const int steps = K / BK, blocks = (steps + 3) / 4, z = blockIdx.y;
    const int z0 = (int)((long)blocks * z / a.kslices);
    const int z1 = (int)((long)blocks * (z + 1) / a.kslices);
    const int b0 = z0 + (z1 - z0) * wave / WAVES, b1 = z0 + (z1 - z0) * (wave + 1) / WAVES;
    const int c0 = 4 * b0, c1 = min(4 * b1, steps);

    f32x16 acc[TB];
#pragma unroll
    for (int f = 0; f < TB; ++f)
#pragma unroll
        for (int e = 0; e < 16; ++e) acc[f][e] = 0.f;

    if (c0 < c1) {
        // (rows past the end: unused)
        const int q = lane & 31;
        const RowPtr rp = GU ? D::rows(q & 2 ? a.up : a.w, min(m0 + 2 * (q >> 2) + (q & 1), M - 1))
                             : D::rows(a.w, min(m0 + q, M - 1));
        const _Float16 *xb[TB];
        const int nblk = (N + 31) / 32;
        // piece(i, h) = piece(i, 0) + h * (piece(0, 1) - piece(0, 0))
        const int hoff = h * (piece<F>(0, 1) - piece<F>(0, 0));
        unsigned pstride[TB]; // halves per piece of the block
#pragma unroll
        for (int b = 0; b < TB; ++b) {
            const int blk = min(b, nblk - 1), c = min(32, N - 32 * blk);
            pstride[b] = 8 * c;
            xb[b] = a.xh + (size_t)blk * 32 * K + min(lane & 31, c - 1) * 8 + hoff * 8 * c;
        }
        typename D::Raw raw[2];
        half8 B[2][TB][2]; // fragments 0, 1 and 2, 3 of a step
        auto load_w = [&](int i, int b) { D::load(raw[i], rp, 4 * min(b, b1 - 1), c1 - 1, h); };
        auto load_b = [&](int s, int c) {
#pragma unroll
            for (int b = 0; b < TB; ++b)
#pragma unroll
                for (int i = 0; i < 2; ++i)
                    B[s][b][i] = *reinterpret_cast<const half8 *>(
                        xb[b] + (8u * c + piece<F>(2 * s + i, 0)) * pstride[b]);
        };
        // (straight-line blocks left only at the loop's end: see px_produce)
        // The next block but one is loaded when its registers are free, so that
        // two are in flight from the start (Q6_K [4096 x 4096] 20 tokens 15.9 ->
        // 14.2 us). Q8_0's blocks, the most bytes and loads (twelve) of the
        // formats, measured faster a block later: [14336 x 4160] 20 tokens 24.1
        // -> 22.6, 64 tokens 28.9 -> 27.9, [4096 x 1088] 20 tokens 9.9 -> 9.2.
        constexpr bool late = F == Q8_0;
        auto block = [&](int d, int b, int n) {
            if (late) load_w(d ^ 1, b + 1);
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                if (F == Q8_0 && u >= n) return;
                const int c = 4 * b + u;
                load_b(1, c);
                half8 w[4];
                D::values(raw[d], u, h, w);
#pragma unroll
                for (int s = 0; s < 2; ++s) {
#pragma unroll
                    for (int i = 0; i < 2; ++i)
#pragma unroll
                        for (int b = 0; b < TB; ++b)
                            acc[b] = __builtin_amdgcn_mfma_f32_32x32x16_f16(w[2 * s + i], B[s][b][i],
                                                                            acc[b], 0, 0, 0);
                    if (s == 0) load_b(0, min(c + 1, c1 - 1));
                }
                if (!late && u == 3) load_w(d, b + 2);
            }
        };
        load_w(0, b0);
        if (!late) load_w(1, b0 + 1);
        load_b(0, c0);
        for (int b = b0;; b += 2) {
            block(0, b, c1 - 4 * b);
            if (b + 1 >= b1) break;
            block(1, b + 1, c1 - 4 * (b + 1));
            if (b + 2 >= b1) break;
        }
    }

    // the waves' sums in wave order: a thread takes four rows of one token of
    // each block
#pragma unroll
    for (int b = 0; b < TB; ++b)
#pragma unroll
        for (int e = 0; e < 4; ++e)
            red[b][wave][e][lane] = make_float4(acc[b][4 * e], acc[b][4 * e + 1],
                                                acc[b][4 * e + 2], acc[b][4 * e + 3]);
    __syncthreads();
    const int m = m0 + (GU ? 4 * wave + 2 * h : 8 * wave + 4 * h);
    if (m >= M) return;
#pragma unroll
    for (int b = 0; b < TB; ++b) {
        const int n = 32 * b + (lane & 31);
        if (n >= N) continue;
        float4 v = red[b][0][wave][lane];
#pragma unroll
        for (int w = 1; w < WAVES; ++w) {
            const float4 p = red[b][w][wave][lane];
            v = make_float4(v.x + p.x, v.y + p.y, v.z + p.z, v.w + p.w);
        }
        const float sc = a.rscale[n];
        v = make_float4(v.x * sc, v.y * sc, v.z * sc, v.w * sc);
        if constexpr (GU) { // gate rows m, m + 1, then up's
            *reinterpret_cast<float2 *>(a.y + (size_t)n * M + m) =
                make_float2(silu_mul(v.x, v.z), silu_mul(v.y, v.w));
            continue;
        }
        const bool split = a.kslices > 1;
        float *y = split ? a.part + ((size_t)z * N + n) * M : a.y + (size_t)n * M;
        const float *rr = !split && a.residual ? a.residual + (size_t)n * M : nullptr;
        if (m + 3 < M && (M & 3) == 0) {
            if (rr) {
                const float4 o = *reinterpret_cast<const float4 *>(rr + m);
                v = make_float4(o.x + v.x, o.y + v.y, o.z + v.z, o.w + v.w);
            }
            *reinterpret_cast<float4 *>(y + m) = v;
        } else {
            const float e4[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
            for (int e = 0; e < 4; ++e)
                if (m + e < M) y[m + e] = rr ? rr[m + e] + e4[e] : e4[e];
        }
    }
}

} // namespace regmm

// One format's launches (each format is its own translation unit).
template <int F> int launch_regmm_format(const regmm::Args &a, int tb, void *stream)
{
    const dim3 grid((a.rtiles + 7) / 8 * 8, a.kslices), block(64 * regmm::WAVES);
    hipStream_t st = (hipStream_t)stream;
    const bool gu = a.up.p0;
    if (tb == 1) {
        if (gu) hipLaunchKernelGGL((regmm::regmm_kernel<F, 1, true>), grid, block, 0, st, a);
        else hipLaunchKernelGGL((regmm::regmm_kernel<F, 1, false>), grid, block, 0, st, a);
        return (int)hipGetLastError();
    }
    if constexpr (F != Q6_K) { // (regmm_fits: one block)
        if (tb == 2) {
            if (gu) hipLaunchKernelGGL((regmm::regmm_kernel<F, 2, true>), grid, block, 0, st, a);
            else hipLaunchKernelGGL((regmm::regmm_kernel<F, 2, false>), grid, block, 0, st, a);
            return (int)hipGetLastError();
        }
    }
    return (int)hipErrorInvalidValue;
}

} // namespace hyq
