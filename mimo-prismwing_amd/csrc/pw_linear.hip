// Block-scaled FP8 projections for decode widths (1..32 activation rows) on gfx950.
//
// Mode A (FP8 weight x f32/bf16 activation, f32 accumulation) follows the reference's
// block_fp8_gemv_parallel_lut_blocked / block_fp8_gemm{1..8}_shared_weight_lut_blocked
// (kernels/block_fp8_gemv.metal:665-703, :751-800, :855-933) and its CPU twin mapped_fp8_gemv
// (src/lib.rs:1272-1309). Mode B (dynamic FP8 activation, block-scaled) follows
// block_fp8_gemm{1..32}_sglang_blockscaled (kernels/block_fp8_gemv.metal:935-1046).
//
// Mode A converts e4m3 to bf16 exactly (v_cvt_scalef32_pk_bf16_fp8) and feeds
// v_mfma_f32_16x16x32_bf16 with the activation rows as the 16-wide N operand; f32 activations are
// split into three bf16 planes (hi + mid + lo == x exactly), so every product is exact and only the
// f32 accumulation order differs from the reference. Mode B feeds the e4m3 codes of weights and
// activations straight into v_mfma_scale_f32_16x16x128_f8f6f4: one instruction is one 128-column
// scale block. The 128x128 block scale (and in mode B the per-token activation scale) is applied to
// the f32 block partial in registers: total += scale * partial. MFMA is used because f32 VALU FMA
// (no packed math) cannot reach 8 TB/s x 8 rows x 2 FLOP/B.
//
//
// The kernel and what bounds it: pw_wide.h.
#include "pw_device.h"
#include "pw_launch.h"
#include "pw_wide.h"

namespace pw {

// ------------------------------------------------------------------ dynamic FP8 quantiser
// dynamic_fp8_quantized_group128 (kernels/block_fp8_gemv.metal:84-137) and its CPU authority
// dynamic_fp8_activations (src/text_endpoint.rs:3008-3051): scale = max(absmax, 1e-10) / 448;
// code = nearest e4m3 of clamp(x/scale). A non-finite input raises FLAG_QUANT_NONFINITE and
// counts as 0 in the group maximum.
// One 128-column group per 16 lanes, 16 groups per 256-thread workgroup (quant_group128_team).
template <typename T>
__global__ __launch_bounds__(256) void quant_group128_kernel(const T *__restrict__ x, uint32_t rows,
                                                             uint32_t K, uint8_t *__restrict__ codes,
                                                             float *__restrict__ scales,
                                                             uint32_t *flags)
{
    const uint32_t group = blockIdx.x * 16 + (threadIdx.x >> 4);
    if (group < rows * (K >> 7))  // whole 16-lane groups leave together
        quant_group128_team<T>(x, group, threadIdx.x & 15, codes, scales, flags);
}

// f32 [n] -> bf16 planes hi [n], mid [n], lo [n] with x == hi + mid + lo.
__global__ __launch_bounds__(256) void split_planes_kernel(const float *__restrict__ x, uint32_t n,
                                                           uint16_t *__restrict__ planes)
{
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n)
        return;
    uint16_t h, m, l;
    split3_bf16(x[i], h, m, l);
    planes[i] = h;
    planes[n + i] = m;
    planes[2 * (size_t)n + i] = l;
}

// ------------------------------------------------------------------------------- launchers
void launch_split_planes(const float *x, uint32_t n, uint16_t *planes, hipStream_t stream)
{
    hipLaunchKernelGGL(split_planes_kernel, dim3((n + 255) / 256), dim3(256), 0, stream, x, n, planes);
}

// Shares of K. Few tiles of a long K leave most of the chip idle while each workgroup takes in the
// batch's rows over the whole K: up to 64 tiles take four shares, up to 128 two, for a second launch
// that adds them, where the rows are enough to pay for it (us, one / two / four shares: 1000 x 8192,
// mode A, one f32 row 10.1 / 9.1 / 8.4, 32 f32 rows 19.0 / 14.5 / 11.6, 16 bf16 rows 9.8 / 8.8 / 8.7,
// one bf16 row 8.2 / 8.6 / 8.5; mode B, 32 rows 16.0 / 12.8 / 11.4; 2000 x 6144, 32 bf16 rows
// 10.1 / 9.4 / 11.9, 8 f32 rows 9.8 / 9.1 / 9.7; 600 x 5120, one f32 row 7.9 / 8.4 / 8.3, 16 f32 rows
// 9.8 / 9.6 / 8.7; 3000 x 8192, 16 f32 rows 14.8 / 19.3 / 18.6).
uint32_t linear_shares(WideX xt, uint32_t W, uint32_t K, uint32_t n_tiles)
{
    const bool pays = xt == WX_F32 ? K >= 6144 || (K >= 5120 && W > 8) : (K >= 8192 && W > 8) || (K >= 6144 && W > 16);
    return pays ? tile_shares(n_tiles) : 1u;
}

// Sixteen waves a workgroup instead of eight. With one tile a CU a wave of eight computes four blocks one
// after another at K = 4096, two of them in flight, and splitting f32 rows into planes costs most of a
// block; sixteen waves have two blocks each. For up to four f32 rows, and for one or two bf16 ones of 8192
// columns, where a wave has whole pairs of blocks (us, eight / sixteen waves, weights in the memory-side
// cache | from HBM: 2048 x 4096, one f32 row 6.0 / 5.8 | 7.5 / 6.6; 4096 x 4096, four f32 rows
// 6.5 / 6.2 | 8.1 / 7.7; 3000 x 8192, one f32 row 9.6 / 9.3 | 11.7 / 10.7, one bf16 row 7.2 / 7.3 |
// 9.4 / 8.6; 3000 x 5120, one f32 row 6.8 / 7.2 | 8.7 / 8.7, 1000 x 6144 7.1 / 7.4 | 7.9 / 7.7; 2048 x 4096,
// one bf16 row 4.8 / 4.9 | 6.1 / 6.1).
static bool sixteen_waves(WideX xt, uint32_t W, uint32_t K, uint32_t KS, uint32_t n_tiles)
{
    return n_tiles <= 256 && K % (KS * 4096) == 0 &&
           (xt == WX_F32 ? W <= 4 : xt == WX_BF16 && W <= 2 && K / KS >= 8192);
}

void launch_linear(WideX xt, const uint8_t *w, const float *s, const ProjTile *tiles, uint32_t n_tiles, const void *x,
                   const float *x_scales, uint32_t W, uint32_t K, float *partial, float *y32, uint16_t *y16, uint32_t N, uint32_t round_f32, hipStream_t stream)
{
    WideArgs args{};
    args.w0 = w;
    args.s0 = s;
    args.tiles = tiles;
    args.n_tiles = n_tiles;
    args.partial = partial;
    args.KS = linear_shares(xt, W, K, n_tiles);
    args.x = x;
    args.x_scales = x_scales;
    args.W = W;
    args.K = K;
    args.N = N;
    args.y_f32 = y32;
    args.y_bf16 = y16;
    args.round_f32 = round_f32;
    const int rt = pick_rt(xt, W, K, n_tiles);
    const int t = timer_begin(xt == WX_CODES ? K_LINEAR_B : K_LINEAR_A, stream);
    const bool aligned = ((uintptr_t)x & 15) == 0;
    if (rt == 1 && sixteen_waves(xt, W, K, args.KS, n_tiles)) {
        if (aligned)
            launch_wide_16<WK_PROJ, true>(xt, args, stream);
        else
            launch_wide_16<WK_PROJ, false>(xt, args, stream);
    } else if (xt == WX_F32 && !aligned)
        launch_wide_unaligned<WK_PROJ, WX_F32>(args, rt, stream);
    else if (xt == WX_BF16 && !aligned)
        launch_wide_unaligned<WK_PROJ, WX_BF16>(args, rt, stream);
    else if (xt == WX_F32)
        launch_wide<WK_PROJ, WX_F32>(args, rt, stream);
    else if (xt == WX_BF16)
        launch_wide<WK_PROJ, WX_BF16>(args, rt, stream);
    else
        launch_wide<WK_PROJ, WX_CODES>(args, rt, stream);
    if (args.KS > 1)
        launch_round_output(partial, args.KS, W * N, y32, y16, !round_f32, nullptr, stream);
    timer_end(t, stream);
}

void launch_quant_group128(const void *x, bool x_f32, uint32_t rows, uint32_t K, uint8_t *codes,
                           float *scales, uint32_t *flags, hipStream_t stream)
{
    const uint32_t groups = rows * (K >> 7);
    const int grid = (int)((groups + 15) / 16);
    const int t = timer_begin(K_QUANT, stream);
    if (x_f32)
        hipLaunchKernelGGL(quant_group128_kernel<float>, dim3(grid), dim3(256), 0, stream,
                           (const float *)x, rows, K, codes, scales, flags);
    else
        hipLaunchKernelGGL(quant_group128_kernel<uint16_t>, dim3(grid), dim3(256), 0, stream,
                           (const uint16_t *)x, rows, K, codes, scales, flags);
    timer_end(t, stream);
}

}  // namespace pw
