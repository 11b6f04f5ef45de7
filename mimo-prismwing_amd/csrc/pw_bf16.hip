// BF16 wide linear for decode widths (attention o_proj [4096 x 8192], LM head [vocab x 4096]):
// y[p, r] = round_bf16(sum_c bf16(W[r, c]) * x[p, c]) in f32, the reference's
// execute_bf16_linear (src/wide_metal_moe.rs:728-834: bf16_gemm8_shared_weight,
// kernels/block_fp8_gemv.metal:358-397, then bf16_round_in_place :219-232) and its CPU twin
// bf16_linear (src/text_endpoint.rs:3347-3380: decode the bf16 tensor, SGEMM, round).
//
// The streaming kernel of pw_wide.h on bf16 weights: f32 rows split into three exact bf16 planes in
// registers, so v_mfma_f32_16x16x32_bf16 forms exact products and accumulates in f32; only the f32
// summation order differs from the reference's. A non-finite result raises FLAG_ROUND_NONFINITE, the
// reference's error bit 32. HBM-bound; against 64-row workgroups of 512 columns each with their
// partials through memory and a reducing launch (us, weights in the memory-side cache): 4096 x 8192
// (67 MB), f32 rows, width 8 18.8 -> 12.7, width 32 42.4 -> 23.2; 16384 x 8192, one row 55.8 -> 40.4.
#include "pw_launch.h"
#include "pw_wide.h"

namespace pw {

// Shares of K. Few tiles of a long K leave most of the chip idle, and one CU's share of the weights
// bounds the launch: up to 64 tiles take four shares, up to 128 two, for a second launch that adds them
// (us, one / two / four / eight shares: 512 x 8192, one f32 row 12.1 / 9.9 / 8.9 / 8.9, 16 bf16 rows
// 12.8 / 10.2 / 8.5 / 8.6; 2048 x 8192, 8 f32 rows 14.0 / 11.1 / 12.1 / 14.9; 3000 x 8192, one
// bf16 row 12.2 / 14.7; 1000 x 5120, 16 f32 rows 11.0 / 10.1 / 9.0; 1000 x 4096, one f32 row 7.9 with
// one share). From 32 bytes of f32 and 48 of bf16 rows a column on, shares pay from K = 4096 (one / two /
// four, weights in the memory-side cache | from HBM: 1000 x 4096, 8 f32 rows 7.3 / 7.0 / 6.6 |
// 8.6 / 8.2 / 7.2, 32 f32 rows 10.6 / 8.8 / 7.6 | 14.9 / 11.5 / 8.9, 32 bf16 rows 7.9 / 7.2 / 6.7 |
// 10.3 / 8.9 / 7.5; 2000 x 4096, 32 bf16 rows 8.2 / 7.7 / 9.6 | 10.7 / 9.6 / 11.1; 1000 x 2048, 32 bf16 rows
// 5.4 / 6.6 / 6.6 | 5.9 / 7.3 / 6.4).
static uint32_t bf16_shares(bool x_f32, uint32_t W, uint32_t K, uint32_t n_tiles)
{
    return K >= (W >= (x_f32 ? 8u : 24u) ? 4096u : 5120u) ? tile_shares(n_tiles) : 1u;
}

// Tiles per workgroup (pw_wide.h's pick_rt for one-byte weights). Twice the weight bytes per tile keep
// one tile ahead while the activations are up to 16 bytes a column, and up to 32 from 513 to 2304 tiles
// (us, one / two / three / four tiles, K = 4096: 1063 tiles, 8 f32 rows 27.6 / 39.6 / 33.0 / 41.4; 2063
// tiles 47.3 / 66.0 / 50.2 / 62.0; 2500 tiles 73.9 / 72.6 / 72.2 / 71.3). Past that a CU holds one
// workgroup of three or four tiles, so the launch takes whole generations of 768 or 1024 tiles: the one
// with the shorter sum of them (1063 tiles, 16 f32 rows 40.9 / 43.5 / 34.9 / 42.8; 2063 tiles
// 71.9 / 74.9 / 53.6 / 64.2; 2500 tiles 100.8 / 80.5 / 77.2 / 76.7; 532 tiles, 32 f32 rows
// 34.0 / 31.3 / 20.9 / 25.2; 848 tiles 43.6 / 32.1 / 38.2 / 26.8). At K = 1024 a wave has one step
// and nothing to overlap: many tiles of 16 to 32 staged bytes a column go by two (1536 tiles, one f32 row
// 14.2 / 11.5 / - / 14.9, 16 bf16 rows 14.4 / 12.3 / 13.4 / 14.8, 4 bf16 rows 11.2 / 11.5 / - / 14.2).
static int bf16_rt(bool x_f32, uint32_t W, uint32_t K, uint32_t n_tiles)
{
    const uint32_t bytes = W * (x_f32 ? 4 : 2);
    if (n_tiles <= 256)
        return 1;
    if (K <= 1024 && n_tiles > 768 && bytes <= 32 && (x_f32 || W > 4))
        return 2;
    if (bytes <= (n_tiles > 512 && n_tiles <= 2304 ? 32u : 16u))
        return 1;
    if (n_tiles <= 512)
        return 2;
    const uint32_t three = (n_tiles + 767) / 768, four = (n_tiles + 1023) / 1024;  // generations
    return 3 * three < 4 * four ? 3 : 4;
}

void launch_bf16_linear(const uint16_t *w, const void *x, bool x_f32, uint32_t W, uint32_t K, uint32_t R, float *partial,
                        float *y32, uint16_t *y16, uint32_t round_f32, uint32_t *flags, hipStream_t stream)
{
    WideArgs args{};
    args.w0 = (const uint8_t *)w;
    args.flags = flags;
    args.n_tiles = (R + 15) / 16;
    args.partial = partial;
    args.KS = bf16_shares(x_f32, W, K, args.n_tiles);
    args.x = x;
    args.W = W;
    args.K = K;
    args.N = R;
    args.y_f32 = y32;
    args.y_bf16 = y16;
    args.round_f32 = round_f32;
    const int rt = bf16_rt(x_f32, W, K, args.n_tiles);
    const int t = timer_begin(K_BF16_LINEAR, stream);
    if (x_f32)
        launch_wide<WK_BF16, WX_F32>(args, rt, stream);
    else
        launch_wide<WK_BF16, WX_BF16>(args, rt, stream);
    if (args.KS > 1)
        launch_round_output(partial, args.KS, W * R, y32, y16, !round_f32, flags, stream);
    timer_end(t, stream);
}

}  // namespace pw
