// Weight::matmul by decoded rows (src/quant.rs:225-237 at batch 1,
// :272-343 at batch >= 2): every row decoded to f32 exactly as the decoder
// does it (an f16 widens without rounding; a Q8_0 value is d * q) and dotted
// with the f32 activations in f32. This serves the F32 and F16 weights (the
// HyV3 router, src/model.rs:223-226, is required F32, and a GGUF file may
// carry either in place of a quantized tensor) and Q8_0 matrices whose width
// is a whole number of 32-value blocks but not of the int8 GEMV's 256-value
// groups or the GEMM's 64-column slices.
//
// Batch 1 is a GEMV, HBM-bound: one wave per row (four rows per 256-thread
// workgroup), each lane streaming 4-value slices of the row with the
// matching float4 of x, four independent fused multiply-adds, then a wave
// reduction. The gate/up form computes silu(g) * u of two rows in the same
// wave. Batch >= 2 runs on the f32 matrix instructions (v_mfma_f32_16x16x4 /
// 32x32x2: f32 products and sums): small outputs, such as a router's, as
// T x T blocks whose K range is split over a workgroup's waves (sixteen for 16
// x 16, eight for 32 x 32), large ones as 64 x 64 tiles with K in steps of 32
// through LDS. The form, and with it the order of the sum, follows the weight's
// shape and the number of rows (gemm_fv).
#include <hip/hip_runtime.h>

#include "hyq_internal.hpp"
#include "hyq_wave.hpp"

namespace hyq {

namespace {

// Value access to one decoded row r of a weight view: elem(k) and, for k a
// multiple of 4, load4(k) (the four values k..k+3, one Q8_0 block).
template <int F> struct Raw;
template <> struct Raw<F32> {
    __device__ static float elem(const WView &w, int cols, int r, int k)
    {
        return reinterpret_cast<const float *>(w.p0)[(size_t)r * cols + k];
    }
    __device__ static float4 load4(const WView &w, int cols, int r, int k)
    {
        return *reinterpret_cast<const float4 *>(reinterpret_cast<const float *>(w.p0) +
                                                 (size_t)r * cols + k);
    }
};
template <> struct Raw<F16> {
    __device__ static float elem(const WView &w, int cols, int r, int k)
    {
        return (float)reinterpret_cast<const _Float16 *>(w.p0)[(size_t)r * cols + k];
    }
    __device__ static float4 load4(const WView &w, int cols, int r, int k)
    {
        typedef _Float16 h4 __attribute__((ext_vector_type(4)));
        const h4 v = *reinterpret_cast<const h4 *>(reinterpret_cast<const _Float16 *>(w.p0) +
                                                   (size_t)r * cols + k);
        return make_float4((float)v.x, (float)v.y, (float)v.z, (float)v.w);
    }
};
// Q8_0 planes: 32 int8 per block, then the blocks' f16 scales
// (decode: d * q, src/quant.rs:2413-2418)
template <> struct Raw<Q8_0> {
    __device__ static float scale(const WView &w, size_t b)
    {
        return (float)reinterpret_cast<const _Float16 *>(w.p1)[b];
    }
    __device__ static float elem(const WView &w, int cols, int r, int k)
    {
        const size_t b = (size_t)r * (cols >> 5) + (k >> 5);
        return scale(w, b) * (float)reinterpret_cast<const int8_t *>(w.p0)[b * 32 + (k & 31)];
    }
    __device__ static float4 load4(const WView &w, int cols, int r, int k)
    {
        const size_t b = (size_t)r * (cols >> 5) + (k >> 5);
        const float d = scale(w, b);
        const uint32_t q = *reinterpret_cast<const uint32_t *>(w.p0 + b * 32 + (k & 31));
        return make_float4(d * (float)(int8_t)(q & 0xff), d * (float)(int8_t)((q >> 8) & 0xff),
                           d * (float)(int8_t)((q >> 16) & 0xff), d * (float)(int8_t)(q >> 24));
    }
};

// The dot of weight row r with x over a wave: lane l takes the 4-value
// slices l, l + 64, ... (VEC: cols % 4 == 0 and x 16-byte aligned), or the
// single values l, l + 64, ... otherwise.
template <int F, bool VEC>
__device__ __forceinline__ float row_dot(const WView &w, int r, const float *x, int cols,
                                         int lane)
{
    float a0 = 0.f, a1 = 0.f, a2 = 0.f, a3 = 0.f;
    if constexpr (VEC) {
        const int n4 = cols >> 2;
        const float4 *x4 = reinterpret_cast<const float4 *>(x);
        for (int c = lane; c < n4; c += 64) {
            const float4 wv = Raw<F>::load4(w, cols, r, 4 * c);
            const float4 xv = x4[c];
            a0 = fmaf(wv.x, xv.x, a0);
            a1 = fmaf(wv.y, xv.y, a1);
            a2 = fmaf(wv.z, xv.z, a2);
            a3 = fmaf(wv.w, xv.w, a3);
        }
    } else {
        for (int c = lane; c < cols; c += 64) a0 = fmaf(Raw<F>::elem(w, cols, r, c), x[c], a0);
    }
    return wave::sum64((a0 + a1) + (a2 + a3));
}

template <int F, bool VEC, bool SILU>
__global__ __launch_bounds__(256) void f32_gemv_kernel(WView w, WView u, int cols,
                                                       const float *__restrict__ x,
                                                       float *__restrict__ y)
{
    const int lane = threadIdx.x & 63;
    const int row = blockIdx.x * 4 + (threadIdx.x >> 6);
    if (row >= w.rows) return;
    const float g = row_dot<F, VEC>(w, row, x, cols, lane);
    if constexpr (SILU) {
        const float v = row_dot<F, VEC>(u, row, x, cols, lane);
        // silu(g) * u, silu(g) = g / (1 + exp(-g)) (src/model.rs:681)
        if (lane == 0) y[row] = (g / (1.0f + expf(-g))) * v;
    } else {
        if (lane == 0) y[row] = g;
    }
}

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

// Values k..k+3 of weight row r, zeros past cols (VEC: cols % 4 == 0).
template <int F, bool VEC>
__device__ __forceinline__ f32x4 weight4(const WView &w, int cols, int r, int k)
{
    const f32x4 z = {0.f, 0.f, 0.f, 0.f};
    if constexpr (VEC) {
        // (an unconditional load, clamped into the row: a load under a
        // condition is waited for at once, and the steps' loads would not
        // be in flight together: F16 [4096 x 4096] at 64 tokens 51.9 us
        // instead of 44.3)
        const float4 q = Raw<F>::load4(w, cols, r, min(k, cols - 4));
        return k < cols ? (f32x4){q.x, q.y, q.z, q.w} : z;
    } else {
        f32x4 v = z;
#pragma unroll
        for (int i = 0; i < 4; ++i)
            if (k + i < cols) v[i] = Raw<F>::elem(w, cols, r, k + i);
        return v;
    }
}
// Values k..k+3 of activation row x, zeros past cols (VEC: also 16-byte
// aligned rows).
template <bool VEC>
__device__ __forceinline__ f32x4 row4(const float *__restrict__ x, int cols, int k)
{
    const f32x4 z = {0.f, 0.f, 0.f, 0.f};
    if constexpr (VEC) {
        const f32x4 q = *reinterpret_cast<const f32x4 *>(x + min(k, cols - 4));
        return k < cols ? q : z;
    } else {
        f32x4 v = z;
#pragma unroll
        for (int i = 0; i < 4; ++i)
            if (k + i < cols) v[i] = x[k + i];
        return v;
    }
}

// A T x T block (T weight rows by T tokens) on the f32 matrix instructions.
// mac() takes one float4 per lane of each operand: lane l holds row l % T and
// the columns 4 (l / T) .. + 3 of a 256 / T column step, four MFMAs (each
// sums one column per lane group; both operands place their columns alike).
// Register e of the result is token l % T and weight row row(e).
template <int T> struct Block;
template <> struct Block<16> {
    typedef f32x4 Acc;
    static constexpr int REGS = 4;
    __device__ static void mac(const f32x4 &w, const f32x4 &x, Acc &acc)
    {
#pragma unroll
        for (int i = 0; i < 4; ++i)
            acc = __builtin_amdgcn_mfma_f32_16x16x4f32(w[i], x[i], acc, 0, 0, 0);
    }
    __device__ static int row(int e, int lane) { return 4 * (lane >> 4) + e; }
};
template <> struct Block<32> {
    typedef f32x16 Acc;
    static constexpr int REGS = 16;
    __device__ static void mac(const f32x4 &w, const f32x4 &x, Acc &acc)
    {
#pragma unroll
        for (int i = 0; i < 4; ++i)
            acc = __builtin_amdgcn_mfma_f32_32x32x2f32(w[i], x[i], acc, 0, 0, 0);
    }
    __device__ static int row(int e, int lane)
    {
        return 8 * (e >> 2) + 4 * (lane >> 5) + (e & 3);
    }
};

// Waves of a split block: the smaller blocks are for outputs that leave most
// CUs idle, where a wave's serial loads are the time.
constexpr int split_waves(int T) { return T == 16 ? 16 : 8; }

// Small outputs: one T x T block per workgroup, its K range in one part per
// wave (operands straight from global memory into registers, a round of U
// steps' loads in flight), the parts added in wave order through LDS. A
// router [64 x 2048] at 64 tokens is 16 workgroups of one short loop each
// instead of one 64 x 64 tile walking K in 128 dependent steps: 360 -> 9.9 us,
// at 500 tokens 339 -> 10.4 us. Bound: each workgroup's 256 KiB of operands
// through one CU's load path, then its MFMAs. F16 weights [4096 x 4096]: 8
// tokens 360 -> 17.5 us, 128 tokens 458 -> 72 us (32 x 32 blocks).
template <int F, bool VEC, int T>
__global__ __launch_bounds__(64 * split_waves(T)) void f32_gemm_split_kernel(
    WView w, int cols, const float *__restrict__ x, int batch, float *__restrict__ y)
{
    using B = Block<T>;
    constexpr int KS = 256 / T; // columns per step
    constexpr int U = T == 16 ? 8 : 4;
    constexpr int SPLIT_WAVES = split_waves(T);
    __shared__ float part[SPLIT_WAVES][T][T + 1]; // [wave][token][row]
    const int t = threadIdx.x, lane = t & 63, wv = t >> 6;
    const int r0 = blockIdx.x * T, b0 = blockIdx.y * T;
    const int r = min(r0 + lane % T, w.rows - 1), b = min(b0 + lane % T, batch - 1);
    const float *xr = x + (size_t)b * cols;
    const int steps = (cols + KS - 1) / KS, per = (steps + SPLIT_WAVES - 1) / SPLIT_WAVES;
    const int s0 = wv * per, s1 = min(steps, s0 + per);
    typename B::Acc acc;
#pragma unroll
    for (int e = 0; e < B::REGS; ++e) acc[e] = 0.f;
    for (int s = s0; s < s1; s += U) {
        f32x4 a[U], v[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            // (steps past the wave's part: columns past the end, zeros)
            const int k = s + u < s1 ? (s + u) * KS + 4 * (lane / T) : cols;
            a[u] = weight4<F, VEC>(w, cols, r, k);
            v[u] = row4<VEC>(xr, cols, k);
        }
        // every load is issued before the first product (the scheduler
        // would otherwise pair each load with its products: the router
        // 11.9 us with eight waves, 10.7 so; 32 x 32 blocks, with more waves, ran 15 % slower so)
        if (T == 16) __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int u = 0; u < U; ++u) B::mac(a[u], v[u], acc);
    }
#pragma unroll
    for (int e = 0; e < B::REGS; ++e) part[wv][lane % T][B::row(e, lane)] = acc[e];
    __syncthreads();
    for (int i = t; i < T * T; i += 64 * SPLIT_WAVES) {
        const int bb = i / T, rr = i % T;
        float v = part[0][bb][rr];
#pragma unroll
        for (int z = 1; z < SPLIT_WAVES; ++z) v += part[z][bb][rr];
        if (b0 + bb < batch && r0 + rr < w.rows) y[(size_t)(b0 + bb) * w.rows + r0 + rr] = v;
    }
}

constexpr int MM_T = 64;  // rows and tokens per workgroup
constexpr int MM_K = 32;  // K step through LDS
constexpr int MM_P = MM_K + 4; // LDS row pitch (floats): float4 reads of 8 rows on 8 bank groups

// Large outputs: 64 x 64 tiles, each of the four waves a 32 x 32 quadrant,
// K in steps of 32 through two LDS buffers, the next step's loads in flight
// under the current one's 16 MFMAs. Bound: the f32 MFMA rate (64 cycles per
// 32 x 32 x 2; F16 weights [14336 x 4096] at 1000 tokens 102 TFLOP/s, 71.5
// with 4 x 4 register tiles of f32 FMAs; [4096 x 4096] at 400 444 -> 178 us).
template <int F, bool VEC>
__global__ __launch_bounds__(256) void f32_gemm_kernel(WView w, int cols,
                                                       const float *__restrict__ x, int batch,
                                                       float *__restrict__ y)
{
    __shared__ __align__(16) float Ws[2][MM_T][MM_P], Xs[2][MM_T][MM_P];
    const int t = threadIdx.x, lane = t & 63, wv = t >> 6;
    const int r0 = blockIdx.x * MM_T, b0 = blockIdx.y * MM_T;
    // loader: thread t takes columns 4 (t % 8) of rows t / 8 and t / 8 + 32
    const int lr = t >> 3, lk = 4 * (t & 7);
    int wr[2];
    const float *xr[2];
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        wr[i] = min(r0 + lr + 32 * i, w.rows - 1);
        xr[i] = x + (size_t)min(b0 + lr + 32 * i, batch - 1) * cols;
    }
    f32x4 a[2], v[2];
    auto fetch = [&](int k0) {
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            a[i] = weight4<F, VEC>(w, cols, wr[i], k0 + lk);
            v[i] = row4<VEC>(xr[i], cols, k0 + lk);
        }
    };
    auto put = [&](int p) {
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            *reinterpret_cast<f32x4 *>(&Ws[p][lr + 32 * i][lk]) = a[i];
            *reinterpret_cast<f32x4 *>(&Xs[p][lr + 32 * i][lk]) = v[i];
        }
    };
    f32x16 acc;
#pragma unroll
    for (int e = 0; e < 16; ++e) acc[e] = 0.f;
    const int ar = 32 * (wv >> 1) + (lane & 31), br = 32 * (wv & 1) + (lane & 31);
    const int kl = 4 * (lane >> 5);
    fetch(0);
    put(0);
    __syncthreads();
    for (int k0 = 0, p = 0; k0 < cols; k0 += MM_K, p ^= 1) {
        const bool more = k0 + MM_K < cols;
        if (more) fetch(k0 + MM_K);
#pragma unroll
        for (int kk = 0; kk < MM_K; kk += 8)
            Block<32>::mac(*reinterpret_cast<const f32x4 *>(&Ws[p][ar][kk + kl]),
                           *reinterpret_cast<const f32x4 *>(&Xs[p][br][kk + kl]), acc);
        if (more) put(p ^ 1); // (last read before the previous barrier)
        __syncthreads();
    }
    const int b = b0 + br;
    if (b >= batch) return;
#pragma unroll
    for (int e = 0; e < 16; ++e) {
        const int r = r0 + 32 * (wv >> 1) + Block<32>::row(e, lane);
        if (r < w.rows) y[(size_t)b * w.rows + r] = acc[e];
    }
}

template <int F>
int gemv_f(WView w, const WView *u, int cols, const float *x, float *y, hipStream_t st)
{
    const dim3 grid((w.rows + 3) / 4), block(256);
    const bool vec = cols % 4 == 0 && (uintptr_t)x % 16 == 0;
    if (u) {
        if (vec) hipLaunchKernelGGL((f32_gemv_kernel<F, true, true>), grid, block, 0, st, w, *u, cols, x, y);
        else hipLaunchKernelGGL((f32_gemv_kernel<F, false, true>), grid, block, 0, st, w, *u, cols, x, y);
    } else {
        if (vec) hipLaunchKernelGGL((f32_gemv_kernel<F, true, false>), grid, block, 0, st, w, w, cols, x, y);
        else hipLaunchKernelGGL((f32_gemv_kernel<F, false, false>), grid, block, 0, st, w, w, cols, x, y);
    }
    return (int)hipGetLastError();
}

// The 64 x 64 tiles where they give every CU one; else 32 x 32 blocks where
// those do, else 16 x 16 blocks (the most workgroups, the most operand reads
// per product): each rule's line is the count below which CUs stay idle. Below
// 512 columns a 16 x 16 block's sixteen waves have too little to split and a CU
// holds one block, so 32 x 32 blocks take those ([300 x 96] F32: 777 rows 15.8
// -> 3.9 us, 64 rows 5.0 -> 3.8; [64 x 252] 64 rows 6.8 -> 3.6), with
// single-value loads, which favour more waves, from 256 columns only past one
// round of 16 x 16 blocks ([64 x 257] 64 rows 6.0 against 7.5; [300 x 257] 250
// rows 10.7 -> 8.0).
// The three sum K in different orders, so the count is of `total` rows: a caller
// that runs them in several passes gives a row the same bits in any of them.
// Between products of different totals a row's last bits may differ ([4096 x
// 4096]: at 33 and at 193 rows).
template <int F, bool VEC>
int gemm_fv(WView w, int cols, const float *x, int batch, int total, float *y, hipStream_t st)
{
    auto grid = [&](int T) { return dim3((w.rows + T - 1) / T, (batch + T - 1) / T); };
    auto count = [&](int T) { return (size_t)grid(T).x * ((total + T - 1) / T); };
    const bool narrow = cols < 512 && (VEC || cols < 256 || count(16) > 256);
    if (count(64) >= 256)
        hipLaunchKernelGGL((f32_gemm_kernel<F, VEC>), grid(64), dim3(256), 0, st, w, cols, x,
                           batch, y);
    else if (narrow || count(32) >= 256)
        hipLaunchKernelGGL((f32_gemm_split_kernel<F, VEC, 32>), grid(32), dim3(64 * split_waves(32)),
                           0, st, w, cols, x, batch, y);
    else
        hipLaunchKernelGGL((f32_gemm_split_kernel<F, VEC, 16>), grid(16), dim3(64 * split_waves(16)),
                           0, st, w, cols, x, batch, y);
    return (int)hipGetLastError();
}

template <int F>
int gemm_f(WView w, int cols, const float *x, int batch, int total, float *y, hipStream_t st)
{
    return cols % 4 == 0 && (uintptr_t)x % 16 == 0
               ? gemm_fv<F, true>(w, cols, x, batch, total, y, st)
               : gemm_fv<F, false>(w, cols, x, batch, total, y, st);
}

} // namespace

int launch_f32_gemv(int fmt, WView w, const WView *up, int cols, const float *x, float *y,
                    void *stream)
{
    hipStream_t st = (hipStream_t)stream;
    if (w.rows <= 0) return 0;
    if (fmt == F32) return gemv_f<F32>(w, up, cols, x, y, st);
    if (fmt == F16) return gemv_f<F16>(w, up, cols, x, y, st);
    if (fmt == Q8_0) return gemv_f<Q8_0>(w, up, cols, x, y, st);
    return (int)hipErrorInvalidValue;
}

int launch_f32_gemm(int fmt, WView w, int cols, const float *x, int batch, int total, float *y,
                    void *stream)
{
    hipStream_t st = (hipStream_t)stream;
    if (w.rows <= 0 || batch <= 0) return 0;
    if (fmt == F32) return gemm_f<F32>(w, cols, x, batch, total, y, st);
    if (fmt == F16) return gemm_f<F16>(w, cols, x, batch, total, y, st);
    if (fmt == Q8_0) return gemm_f<Q8_0>(w, cols, x, batch, total, y, st);
    return (int)hipErrorInvalidValue;
}

} // namespace hyq
