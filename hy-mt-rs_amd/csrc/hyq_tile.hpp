// Building blocks of the f16-MFMA GEMMs on gfx950 (batched matmul,
// Weight::matmul batch >= 2, src/quant.rs:272-344, and the MoE expert
// products, src/model.rs:699-725).
//
// A workgroup owns up to BM = 128 weight rows by up to 256 tokens and walks K
// in BK = 64 steps: producer waves fetch the packed bytes of the next steps
// and dequantize a step's 64 columns into one of two LDS buffers with the
// reference decoder's f32 arithmetic (decode_unchecked, src/quant.rs:
// 2405-2486) and one f32->f16 rounding, while consumer waves multiply the
// other with v_mfma_f32_32x32x16_f16, in f32 (k_loop_px).
// LDS rows are padded to 72 halves (144 bytes), so the 16-byte fragment
// reads of 8 consecutive rows fall on 8 distinct 4-bank windows.
#pragma once

#include <hip/hip_runtime.h>

#include "hyq_decode.hpp"
#include "hyq_groups.hpp"

namespace hyq {
namespace tile {

typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef _Float16 half2v __attribute__((ext_vector_type(2)));
typedef float float2v __attribute__((ext_vector_type(2)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

constexpr int BM = 128, BN = 128, BK = 64, LDK = BK + 8;
constexpr int TILE_HALVES = BM * LDK; // one LDS operand buffer (BM == BN)

__device__ __forceinline__ float h2f(uint32_t bits16)
{
    _Float16 h;
    uint16_t b = (uint16_t)bits16;
    __builtin_memcpy(&h, &b, 2);
    return (float)h;
}

__device__ __forceinline__ uint32_t byte_of(uint32_t dw, int i) { return (dw >> (8 * i)) & 0xffu; }

// ---------------------------------------------------------------------------
// Per-format dequantization of a row's weights by two lanes, 32 of every 64
// columns (a step) each: half h holds the columns c0(h) .. c0(h) + 15 and
// c1(h) .. c1(h) + 15 of a step (which 32 a half takes depends on the format;
// the two halves of a row cover all 64). load() only issues global loads from
// the row's plane bases (RowPtr, computed once per thread), for the four steps
// s .. s + 3 at once: a row's bytes of 256 columns are one 128-byte line or
// two, which a load per step would fetch from L2 again at each (Q4_K
// [14336 x 4096] at 512 tokens moved 66 KB per step and CU so, of which 37
// were its own). s is a multiple of 4 but for Q8_0, whose rows may end within
// the four: their steps past `last` read it again. values() does the
// arithmetic from registers, for step u of the four.
//
// Every value is formed as one fma whose exact result is the decoder's
// exact value, so the f32 result is bit-identical to decode_unchecked
// (src/quant.rs:2405-2486), then rounded once to f16: the packed codes are
// widened with v_cvt_f32_ubyteN (byte n of a dword to f32) and offsets are
// folded into the fma's addend (q - 32 as s*q + (-32 s), int8 q as
// d*(q + 128) + (-128 d), 2c - 3 as 2d*c + (-3d)). The products in those
// addends and multipliers are exact in f32 (at most 24 significant bits).
// ---------------------------------------------------------------------------
struct RowPtr {
    const uint8_t *p0, *p1, *p2;
};

__device__ __forceinline__ RowPtr row_ptr(const WView &w, int F_p0, int F_p1, int F_p2, int row)
{
    const size_t b = (size_t)row * w.nb;
    return RowPtr{w.p0 + b * F_p0, w.p1 + b * F_p1, w.p2 + b * F_p2};
}

// byte i of x as f32 (v_cvt_f32_ubyte{i})
__device__ __forceinline__ float ub(uint32_t x, int i) { return (float)((x >> (8 * i)) & 0xffu); }

// Eight codes (the bytes of lo, then of hi) as f16(d * q + o).
__device__ __forceinline__ half8 deq8(uint32_t lo, uint32_t hi, float d, float o)
{
    // (the dwords as they are: else each byte is first extracted on its own,
    // instead of by its v_cvt_f32_ubyteN)
    asm("" : "+v"(lo), "+v"(hi));
    half8 r;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const uint32_t x = i < 2 ? lo : hi;
        const int j = 2 * (i & 1);
        const half2v p = __builtin_convertvector((float2v){__builtin_fmaf(d, ub(x, j), o),
                                                           __builtin_fmaf(d, ub(x, j + 1), o)},
                                                 half2v);
        r[2 * i] = p[0];
        r[2 * i + 1] = p[1];
    }
    return r;
}

template <int F> struct Deq;

// The values rounded to f16 at their columns of dst (an LDS row): the half's
// columns c0 .. (PART 0), c1 .. (PART 1) or both (PART -1).
template <int F, int PART>
__device__ __forceinline__ void convert(const typename Deq<F>::Raw &r, int u, int h,
                                        _Float16 *dst)
{
    half8 w[4];
    Deq<F>::values(r, u, h, w);
    half8 *p0 = reinterpret_cast<half8 *>(dst + Deq<F>::c0(h));
    half8 *p1 = reinterpret_cast<half8 *>(dst + Deq<F>::c1(h));
    if constexpr (PART != 1) {
        p0[0] = w[0];
        p0[1] = w[1];
    }
    if constexpr (PART != 0) {
        p1[0] = w[2];
        p1[1] = w[3];
    }
}

// Q4_K (decode_unchecked, src/quant.rs:2437-2461): byte l of a 64-weight
// chunk holds weight l (low nibble, sub-block 2c) and 32 + l (high nibble,
// sub-block 2c+1); value = (d*s_j)*q - (dmin*m_j). Half h takes bytes
// 16h..16h+15, i.e. columns 16h.. and 32+16h...
template <> struct Deq<Q4_K> {
    struct Raw {
        u32x4 q[4], meta;
    };
    __device__ static constexpr int c0(int h) { return 16 * h; }
    __device__ static constexpr int c1(int h) { return 32 + 16 * h; }
    __device__ __forceinline__ static RowPtr rows(const WView &w, int row)
    {
        return row_ptr(w, 128, 16, 0, row);
    }
    __device__ __forceinline__ static void load(Raw &r, const RowPtr &p, int s, int, int h)
    {
        const int blk = s >> 2;
        r.meta = *reinterpret_cast<const u32x4 *>(p.p1 + blk * 16);
#pragma unroll
        for (int c = 0; c < 4; ++c)
            r.q[c] = *reinterpret_cast<const u32x4 *>(p.p0 + blk * 128 + 32 * c + 16 * h);
    }
    __device__ __forceinline__ static void scale_min(const u32x4 &meta, int j, int &s, int &m)
    {
        auto sc = [&](int i) -> int {
            const uint32_t dw = i < 4 ? meta.y : i < 8 ? meta.z : meta.w;
            return (int)byte_of(dw, i & 3);
        };
        if (j < 4) {
            s = sc(j) & 63;
            m = sc(j + 4) & 63;
        } else {
            s = (sc(j + 4) & 15) | ((sc(j - 4) >> 6) << 4);
            m = (sc(j + 4) >> 4) | ((sc(j) >> 6) << 4);
        }
    }
    __device__ __forceinline__ static void values(const Raw &r, int u, int h, half8 (&w)[4])
    {
        const int c = u;
        const float d = h2f(r.meta.x & 0xffffu), dmin = h2f(r.meta.x >> 16);
        int s0, m0, s1, m1;
        scale_min(r.meta, 2 * c, s0, m0);
        scale_min(r.meta, 2 * c + 1, s1, m1);
        const float da = d * (float)s0, nm1a = -(dmin * (float)m0);
        const float db = d * (float)s1, nm1b = -(dmin * (float)m1);
        const uint32_t q[4] = {r.q[u].x, r.q[u].y, r.q[u].z, r.q[u].w};
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const uint32_t x = q[2 * i], y = q[2 * i + 1];
            w[i] = deq8(x & 0x0F0F0F0Fu, y & 0x0F0F0F0Fu, da, nm1a);
            w[2 + i] = deq8((x >> 4) & 0x0F0F0F0Fu, (y >> 4) & 0x0F0F0F0Fu, db, nm1b);
        }
    }
};

// Q6_K (src/quant.rs:2462-2483): in a 128-weight chunk, weight p*32+hf*16+i
// has low bits from ql[(p&1)*32 + hf*16 + i] (nibble p>>1) and high bits
// from qh[hf*16 + i] (bits 2p); value = (d*sc[2p+hf]) * (q - 32). A 64-slice
// holds planes p0, p0+1 (p0 even); half h takes plane p0 + h.
template <> struct Deq<Q6_K> {
    struct Raw {
        u32x4 l[2][2], g[2][2], sc; // by 128-weight chunk
        uint32_t d;
    };
    __device__ static constexpr int c0(int h) { return 32 * h; }
    __device__ static constexpr int c1(int h) { return 32 * h + 16; }
    __device__ __forceinline__ static RowPtr rows(const WView &w, int row)
    {
        return row_ptr(w, 192, 16, 2, row);
    }
    __device__ __forceinline__ static void load(Raw &r, const RowPtr &p, int s, int, int h)
    {
        const int blk = s >> 2;
        const uint8_t *base = p.p0 + blk * 192;
        r.sc = *reinterpret_cast<const u32x4 *>(p.p1 + blk * 16);
        r.d = *reinterpret_cast<const uint16_t *>(p.p2 + blk * 2);
#pragma unroll
        for (int c = 0; c < 2; ++c)
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                r.l[c][i] = *reinterpret_cast<const u32x4 *>(base + c * 64 + 32 * h + 16 * i);
                r.g[c][i] = *reinterpret_cast<const u32x4 *>(base + 128 + c * 32 + 16 * i);
            }
    }
    __device__ __forceinline__ static void values(const Raw &r, int u, int h, half8 (&w)[4])
    {
        const int chunk = u >> 1, pl = 2 * (u & 1) + h;
        const float d = h2f(r.d);
        // scales 2 pl and 2 pl + 1 of the chunk's eight
        const uint32_t sc = r.sc[2 * chunk + (u & 1)] >> (16 * h);
        const float s0 = d * (float)(int8_t)(sc & 0xff), s1 = d * (float)(int8_t)(sc >> 8);
        const float o0 = -32.f * s0, o1 = -32.f * s1;
        const u32x4 &l0 = r.l[chunk][0], &l1 = r.l[chunk][1], &g0 = r.g[chunk][0],
                    &g1 = r.g[chunk][1];
        const uint32_t ql[8] = {l0.x, l0.y, l0.z, l0.w, l1.x, l1.y, l1.z, l1.w};
        const uint32_t qh[8] = {g0.x, g0.y, g0.z, g0.w, g1.x, g1.y, g1.z, g1.w};
        // (pl >> 1 is the step's parity)
        const int lsh = (u & 1) * 4, hsh = 2 * pl;
        auto codes = [&](int i) {
            return ((ql[i] >> lsh) & 0x0F0F0F0Fu) | (((qh[i] >> hsh) & 0x03030303u) << 4);
        };
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            w[i] = deq8(codes(2 * i), codes(2 * i + 1), s0, o0);
            w[2 + i] = deq8(codes(4 + 2 * i), codes(5 + 2 * i), s1, o1);
        }
    }
};

// Q8_0 (src/quant.rs:2409-2414): value = d * q; half h takes the 32-block h.
template <> struct Deq<Q8_0> {
    struct Raw {
        u32x4 a[4], b[4];
        uint32_t d[4];
    };
    __device__ static constexpr int c0(int h) { return 32 * h; }
    __device__ static constexpr int c1(int h) { return 32 * h + 16; }
    __device__ __forceinline__ static RowPtr rows(const WView &w, int row)
    {
        return row_ptr(w, 32, 2, 0, row);
    }
    __device__ __forceinline__ static void load(Raw &r, const RowPtr &p, int s, int last, int h)
    {
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            const int blk = 2 * min(s + c, last) + h;
            r.a[c] = *reinterpret_cast<const u32x4 *>(p.p0 + blk * 32);
            r.b[c] = *reinterpret_cast<const u32x4 *>(p.p0 + blk * 32 + 16);
            r.d[c] = *reinterpret_cast<const uint16_t *>(p.p1 + blk * 2);
        }
    }
    __device__ __forceinline__ static void values(const Raw &r, int u, int h, half8 (&w)[4])
    {
        const float d = h2f(r.d[u]), o = -128.f * d;
        const u32x4 &a = r.a[u], &b = r.b[u];
        const uint32_t q[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
#pragma unroll
        for (int i = 0; i < 4; ++i) // q + 128
            w[i] = deq8(q[2 * i] ^ 0x80808080u, q[2 * i + 1] ^ 0x80808080u, d, o);
    }
};

// Q2_0C (src/quant.rs:2415-2422): value = (2c - 3) * d. The device plane
// keeps a 64-weight unit in 16 bytes with weight 16k+i in bits 2k of byte i;
// half h takes k = 2h and 2h+1 (columns 32h..32h+31).
template <> struct Deq<Q2_0C> {
    struct Raw {
        u32x4 c[4];
        uint32_t d;
    };
    __device__ static constexpr int c0(int h) { return 32 * h; }
    __device__ static constexpr int c1(int h) { return 32 * h + 16; }
    __device__ __forceinline__ static RowPtr rows(const WView &w, int row)
    {
        return row_ptr(w, 128, 2, 0, row);
    }
    __device__ __forceinline__ static void load(Raw &r, const RowPtr &p, int s, int, int)
    {
        r.d = *reinterpret_cast<const uint16_t *>(p.p1 + (s >> 3) * 2);
#pragma unroll
        for (int c = 0; c < 4; ++c)
            r.c[c] = *reinterpret_cast<const u32x4 *>(p.p0 + (s + c) * 16);
    }
    __device__ __forceinline__ static void values(const Raw &r, int u, int h, half8 (&w)[4])
    {
        const float d = h2f(r.d), d2 = 2.f * d, o = -3.f * d;
        const uint32_t cw[4] = {r.c[u].x, r.c[u].y, r.c[u].z, r.c[u].w};
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int k = 0; k < 2; ++k)
                w[2 * k + i] = deq8((cw[2 * i] >> (4 * h + 2 * k)) & 0x03030303u,
                                    (cw[2 * i + 1] >> (4 * h + 2 * k)) & 0x03030303u, d2, o);
    }
};

// STQ1_0 (src/quant.rs:1086-1123, 2423-2430): 64-weight chunk c holds 16
// groups; digit p of group gg is column p*16 + gg, value (digit - 1) * d with
// the digit read from the codebook entry of (sign << 4 | nibble). Half h
// takes digits 2h and 2h+1. Device planes as in hyq_internal.hpp: groups
// 4j..4j+3 have their nibbles in bytes of dword j/2 (high nibbles for odd j)
// and their signs at bits (c%2)*4 + j + 8t of the chunk pair's sign dword.
template <> struct Deq<STQ1_0> {
    struct Raw {
        u32x4 nib[2];
        uint32_t s[2], d;
    };
    __device__ static constexpr int c0(int h) { return 32 * h; }
    __device__ static constexpr int c1(int h) { return 32 * h + 16; }
    __device__ __forceinline__ static RowPtr rows(const WView &w, int row)
    {
        return row_ptr(w, 32, 8, 2, row);
    }
    __device__ __forceinline__ static void load(Raw &r, const RowPtr &p, int s, int, int)
    {
        const int blk = s >> 2;
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            r.nib[i] = *reinterpret_cast<const u32x4 *>(p.p0 + blk * 32 + 16 * i);
            r.s[i] = *reinterpret_cast<const uint32_t *>(p.p1 + blk * 8 + 4 * i);
        }
        r.d = *reinterpret_cast<const uint16_t *>(p.p2 + blk * 2);
    }
    __device__ __forceinline__ static void values(const Raw &r, int u, int h, half8 (&w)[4])
    {
        const int c = u;
        const float d = h2f(r.d), o = -d;
        const uint32_t nb[2] = {r.nib[c >> 1][2 * (c & 1)], r.nib[c >> 1][2 * (c & 1) + 1]};
        uint32_t e[4]; // the groups' codebook entries, four per dword
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const uint32_t nibs = (nb[j >> 1] >> (4 * (j & 1))) & 0x0F0F0F0Fu;
            const uint32_t sb = ((r.s[c >> 1] >> ((c & 1) * 4 + j)) & 0x01010101u) << 4;
            e[j] = GroupSTQ::lut(nibs | sb) >> (4 * h);
        }
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int k = 0; k < 2; ++k)
                w[2 * k + i] = deq8((e[2 * i] >> (2 * k)) & 0x03030303u,
                                    (e[2 * i + 1] >> (2 * k)) & 0x03030303u, d, o);
    }
};

__device__ __forceinline__ float silu_mul(float g, float u)
{
    // (g / (1 + exp(-g))) * u, DenseFfn::forward (src/model.rs:680-682)
    return (g / (1.0f + expf(-g))) * u;
}

// v_mfma 32x32 output layout: register e of a block holds row
// 8*(e/4) + 4*(lane/32) + e%4 and column lane%32 of the block.
__device__ __forceinline__ int acc_row_in_block(int e)
{
    return 8 * (e >> 2) + 4 * ((threadIdx.x & 63) >> 5) + (e & 3);
}
// ---------------------------------------------------------------------------
// The K loop of every tile kernel: 512 threads, waves 0-3 (one per SIMD)
// dequantize the weights, waves 4-7 (the other wave of each SIMD) multiply.
//
// LDS holds only the dequantized weights: two buffers of BM rows x BK columns.
// The activations come in fragment order (hyq_f16rows.hpp) straight into the
// consumers' registers, a contiguous KiB per load of a full 32-token block.
// A shape C has NP = 4 producer and NC consumer waves, WR of which share the tokens and split the rows, each
// holding C::RB row blocks by C::CB token blocks of 32 (WR = 1: 4 x 2 blocks,
// a tile of 128 rows by 256 tokens, or RB = 3, 96, or RB = 2, 64 rows; WR = 2:
// 2 x CB blocks, 128 rows by 64 CB tokens). Wave (wr, wc) takes the token blocks wc, wc + WC,
// ..., and only those that hold tokens of the tile (cnt), so a partial tile
// costs its own blocks. Per MFMA a wave reads 1/CB KiB from LDS and 1/RB from
// L1/L2.
//
// What bounds it: the consumers' MFMAs and, where few token blocks share a
// dequantized weight, the producers' conversion (about 3.2 VALU instructions
// per weight). Both are kept from waiting:
//  - the packed bytes of the next four steps are in flight in the producers'
//    registers;
//  - the consumers are software-pipelined, held by scheduling barriers: the
//    weight fragments of the next 16 columns are read from LDS before the
//    current ones' MFMAs (the compiler else keeps two in flight, each pair
//    of MFMAs waiting for its own), the tokens NS steps ahead into the
//    registers just consumed (unconditionally, past the end the last step
//    again: a branch there made every other step wait for the loads it had
//    just issued);
//  - a step's buffer is done with once its last fragments are in registers,
//    so its barrier comes before their MFMAs and the next buffer's first reads
//    run under them.
//
// wsrc(lrow, view, row): the weight view and row that LDS row lrow
// dequantizes (any of the view's for a row past the end, whose sums nobody
// writes); xt: the operand run of the tile's first
// token, cnt >= 1 its tokens; arow(i): the first LDS row of the wave's row
// block i. The loop covers columns [kbase, kbase + klen) of K (multiples of
// the format's block and of BK). Every output element sees the same operands
// in the same k order in every form: bit-identical results.
// ---------------------------------------------------------------------------
constexpr int PX_LDS = 2 * TILE_HALVES;

template <int F, int ROWS, int PART, class WSrc>
__device__ __forceinline__ void px_produce(const WSrc &wsrc, int steps, int kbase, _Float16 *lds)
{
    using D = Deq<F>;
    // (64 rows: two threads to a weight's 32 columns, one per PART)
    const int t = threadIdx.x & (ROWS > 64 ? 255 : 127), lrow = t >> 1, h = t & 1;
    if (ROWS < BM && __builtin_amdgcn_readfirstlane(lrow) >= ROWS) { // (by wave)
        for (int s = 0; s <= steps; ++s) __syncthreads();
        return;
    }
    WView wv{};
    int row = 0;
    wsrc(lrow, wv, row);
    const RowPtr rp = D::rows(wv, row);
    // two 256-column blocks: one is dequantized while the next is loaded (the
    // last again, unused, past the end), in straight-line code: a load under
    // a condition, or a loop left in its middle and entered again, makes the
    // compiler's counted waits wait for the loads just issued
    typename D::Raw raw[2];
    const int s0 = kbase / BK, blocks = (steps + 3) / 4;
    auto fetch = [&](int b, int i) {
        D::load(raw[i], rp, s0 + 4 * min(b, blocks - 1), s0 + steps - 1, h);
    };
    fetch(0, 0);
    for (int bb = 0;; bb += 2) {
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            fetch(bb + i + 1, i ^ 1);
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                convert<F, PART>(raw[i], u, h, lds + (u & 1) * TILE_HALVES + lrow * LDK);
                __syncthreads();
                // (only Q8_0's rows may end within a block)
                if ((u == 3 || F == Q8_0) && 4 * (bb + i) + u + 1 >= steps) {
                    __syncthreads();
                    return;
                }
            }
        }
    }
}

template <int RB, int CB, int J, int NS, class ARow>
__device__ __forceinline__ void px_consume(const _Float16 *xt, int cnt, int K, int wc, int WC,
                                           const ARow &arow, int steps, int kbase,
                                           const _Float16 *lds, f32x16 (&acc)[RB][CB])
{
    const int lane = threadIdx.x & 63, r = lane & 31, h = lane >> 5;
    const _Float16 *xb[J];
    unsigned stride[J]; // halves per 16 columns of the block
#pragma unroll
    for (int j = 0; j < J; ++j) {
        const int b = j * WC + wc, c = min(32, cnt - 32 * b);
        xb[j] = xt + (size_t)32 * b * K + (size_t)kbase * c + (h * c + min(r, c - 1)) * 8;
        stride[j] = 16 * c;
    }
    half8 B[NS][4][J], a[2][RB];
    auto loadB = [&](int s, int set, int kk) {
        const unsigned k16 = 4u * min(s, steps - 1) + kk;
#pragma unroll
        for (int j = 0; j < J; ++j)
            B[set][kk][j] = *reinterpret_cast<const half8 *>(xb[j] + k16 * stride[j]);
    };
    auto loadA = [&](int set, const _Float16 *Ws, int kk) {
#pragma unroll
        for (int i = 0; i < RB; ++i)
            a[set][i] = *reinterpret_cast<const half8 *>(Ws + (arow(i) + r) * LDK + 16 * kk + 8 * h);
    };
#pragma unroll
    for (int p = 0; p < NS; ++p)
#pragma unroll
        for (int kk = 0; kk < 4; ++kk) {
            loadB(p, p, kk);
            __builtin_amdgcn_sched_barrier(0);
        }
    __syncthreads();
    loadA(0, lds, 0);
    auto step = [&](int s, int p) {
        const _Float16 *Ws = lds + (p & 1) * TILE_HALVES, *Wn = lds + (p & 1 ^ 1) * TILE_HALVES;
        const int set = p & (NS - 1);
#pragma unroll
        for (int kk = 0; kk < 4; ++kk) {
            if (kk < 3) {
                loadA((kk + 1) & 1, Ws, kk + 1);
            } else {
                __syncthreads();
                loadA(0, Wn, 0);
            }
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int i = 0; i < RB; ++i)
#pragma unroll
                for (int j = 0; j < J; ++j)
                    acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a[kk & 1][i], B[set][kk][j],
                                                                       acc[i][j], 0, 0, 0);
            __builtin_amdgcn_sched_barrier(0);
            loadB(s + NS, set, kk);
        }
    };
    // (U steps a round, by the rings of both; the last ones singly)
    constexpr int U = NS > 2 ? NS : 2;
    int s = 0;
    for (; s + U <= steps; s += U) {
#pragma unroll
        for (int d = 0; d < U; ++d) step(s + d, d);
    }
#pragma unroll
    for (int d = 0; d + 1 < U; ++d)
        if (s + d < steps) step(s + d, d);
}

// acc[i][j]: row block arow(i), token block j * WC + wc of the tile. Returns
// false for the producers, which hold no sums.
template <int F, class C, class WSrc, class ARow>
__device__ __forceinline__ bool k_loop_px(const WSrc &wsrc, const ARow &arow, const _Float16 *xt,
                                          int cnt, int K, int kbase, int klen, _Float16 *lds,
                                          f32x16 (&acc)[C::RB][C::CB])
{
    constexpr int RB = C::RB, CB = C::CB, NS = C::NS, WC = C::NC / C::WR;
    static_assert(32 * C::WR * RB <= BM && NS >= 1 && NS <= 2 && CB <= 3 &&
                      C::NP == 4,
                  "tile shape");
    const int steps = klen / BK, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    if (wave < C::NP) {
        constexpr int ROWS = 32 * C::WR * RB;
        if (ROWS > 64) px_produce<F, ROWS, -1>(wsrc, steps, kbase, lds);
        else if (wave < 2) px_produce<F, ROWS, 0>(wsrc, steps, kbase, lds);
        else px_produce<F, ROWS, 1>(wsrc, steps, kbase, lds);
        return false;
    }
    const int wc = (wave - C::NP) % WC;
#pragma unroll
    for (int i = 0; i < RB; ++i)
#pragma unroll
        for (int j = 0; j < CB; ++j)
#pragma unroll
            for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.f;
    // this wave's token blocks; both roles pass 1 + steps barriers
    const int nj = ((cnt + 31) / 32 - wc + WC - 1) / WC;
    if (nj >= CB) {
        px_consume<RB, CB, CB, NS>(xt, cnt, K, wc, WC, arow, steps, kbase, lds, acc);
    } else if (CB > 2 && nj == 2) {
        px_consume<RB, CB, 2 < CB ? 2 : 1, NS>(xt, cnt, K, wc, WC, arow, steps, kbase, lds, acc);
    } else if (CB > 1 && nj == 1) {
        // (one block leaves the registers for four steps ahead, and its steps,
        // of half the MFMAs or less, need them)
        px_consume<RB, CB, 1, 4>(xt, cnt, K, wc, WC, arow, steps, kbase, lds, acc);
    } else {
        for (int s = 0; s <= steps; ++s) __syncthreads();
    }
    return true;
}

} // namespace tile
} // namespace hyq
