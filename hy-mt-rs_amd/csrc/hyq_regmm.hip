// Which shapes the few-token products of hyq_regmm_impl.hpp take, and their
// launch by format.
#include <hip/hip_runtime.h>

#include "hyq_regmm_impl.hpp"

namespace hyq {

extern template int launch_regmm_format<Q2_0C>(const regmm::Args &, int, void *);
extern template int launch_regmm_format<STQ1_0>(const regmm::Args &, int, void *);
extern template int launch_regmm_format<Q4_K>(const regmm::Args &, int, void *);
extern template int launch_regmm_format<Q6_K>(const regmm::Args &, int, void *);
extern template int launch_regmm_format<Q8_0>(const regmm::Args &, int, void *);

// Up to one or two 32-token blocks, so one workgroup per row tile: past them
// the weights are dequantized again per 64 tokens and the LDS engine is
// faster (Q4_K [14336 x 4096] at 128 tokens 47.7 against 38 us). Q6_K's second
// block does not fit the registers (spilled, [4096 x 14336] at 64 tokens 66
// against 40 us), and its widest weights, whose row tiles leave a CU one
// workgroup of four waves, are faster in the engine's producers ([4096 x
// 14336] at 30 tokens 36.5 against 28.7 us; [14336 x 4096] 25.3 against 26.7,
// [2048 x 2048] 13.5 against 14.5). At least four 64-column steps per wave: a
// narrower weight leaves the waves that split its columns without work to
// overlap.
bool regmm_fits(int fmt, int cols, int batch)
{
    return batch >= 2 && batch <= (fmt == Q6_K ? 32 : 64) && cols % tile::BK == 0 &&
           cols / tile::BK >= 4 * regmm::WAVES && (fmt != Q6_K || cols < 8192);
}

// K slices across workgroups, where the row tiles leave CUs without one: to
// about one workgroup per CU, at least six steps per wave (the sum's launch
// costs 3.5 us: Q2_0C [2048 x 6144] at 21 tokens 16.4 us in one slice, 14.0
// in four; [6144 x 2048] 10.0 in one, 12.6 in two). A rule on the weight's
// shape only, so that a token's result does not depend on the batch.
int regmm_kslices(int rows, int cols)
{
    if (rows % 4) return 1;
    const int tiles = (rows + 31) / 32, per = cols / tile::BK / regmm::WAVES;
    int ks = 1;
    while (ks < 4 && tiles * ks * 2 <= 256 && per / (2 * ks) >= 6) ks *= 2;
    return ks;
}

// What the kernels take: regmm_fits, and a single row, which a pass may leave
// over of a prompt that takes this form.
static bool launches(int fmt, int cols, int batch)
{
    return batch >= 1 && regmm_fits(fmt, cols, batch < 2 ? 2 : batch);
}

static int launch_format(int fmt, const regmm::Args &a, int tb, void *stream)
{
    switch (fmt) {
    case Q2_0C: return launch_regmm_format<Q2_0C>(a, tb, stream);
    case STQ1_0: return launch_regmm_format<STQ1_0>(a, tb, stream);
    case Q4_K: return launch_regmm_format<Q4_K>(a, tb, stream);
    case Q6_K: return launch_regmm_format<Q6_K>(a, tb, stream);
    case Q8_0: return launch_regmm_format<Q8_0>(a, tb, stream);
    default: return (int)hipErrorInvalidValue;
    }
}

int launch_regmm(int fmt, WView w, int cols, const _Float16 *xh, const float *rscale, int batch,
                 float *y, const float *residual, void *stream, int kslices, float *part)
{
    if (!launches(fmt, cols, batch) || w.rows <= 0 || kslices < 1 || (kslices > 1 && !part))
        return (int)hipErrorInvalidValue;
    const int tb = batch > 32 ? 2 : 1;
    regmm::Args a{};
    a.w = w;
    a.y = y;
    a.residual = residual;
    a.rows = w.rows;
    a.rtiles = (w.rows + 31) / 32;
    a.K = cols;
    a.N = batch;
    a.kslices = kslices;
    a.xh = xh;
    a.rscale = rscale;
    a.part = part;
    const int rc = launch_format(fmt, a, tb, stream);
    if (rc || kslices == 1) return rc;
    return launch_gemm_reduce(part, kslices, (size_t)batch * w.rows, residual, y, stream);
}

int launch_regmm_gate_up(int fmt, WView gate, WView up, int cols, const _Float16 *xh,
                         const float *rscale, int batch, float *h, void *stream)
{
    if (!launches(fmt, cols, batch) || gate.rows <= 0 || gate.rows % 2)
        return (int)hipErrorInvalidValue;
    const int tb = batch > 32 ? 2 : 1;
    regmm::Args a{};
    a.w = gate;
    a.up = up;
    a.y = h;
    a.rows = gate.rows;
    a.rtiles = (gate.rows + 15) / 16;
    a.K = cols;
    a.N = batch;
    a.kslices = 1;
    a.xh = xh;
    a.rscale = rscale;
    return launch_format(fmt, a, tb, stream);
}

} // namespace hyq
