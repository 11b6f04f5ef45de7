// One expert's forward (the complete expert, the dense MLP of a non-routed layer) for 1..32 rows as
// streaming projections (pw_wide.h): gate and up with the SwiGLU in one launch, then down.
#include "pw_launch.h"
#include "pw_wide.h"

namespace pw {

// K shares of the down. A long K over few output rows makes a workgroup of 16 rows read W whole rows
// of activations for 16 rows of weights; two shares of 32-row workgroups halve that for a second
// launch that adds the shares (us of a whole expert, one / two / four shares, K = 16384 over 4096
// rows: f32 hidden, width 8 49.1 / 48.5 / 51.0, width 16 53.8 / 51.2 / 52.0, width 32
// 71.5 / 62.2 / 64.5; codes, width 16 52.4 / 53.1 / 56.0, width 32 61.4 / 58.8 / 60.5; K = 2048 one
// share is best at every width, 16.6 / 17.3 / 18.1 at width 32).
// Up to 128 tiles follow the projections' rule, so that mode B's forward stays the same as its separate
// calls, bit for bit.
static uint32_t down_shares(bool codes, uint32_t W, uint32_t K, uint32_t n_tiles)
{
    if (n_tiles <= 128)
        return linear_shares(codes ? WX_CODES : WX_F32, W, K, n_tiles);
    return n_tiles <= 256 && (uint64_t)K * W >= (codes ? 20u : 12u) * 16384u ? 2u : 1u;
}

void launch_expert_gateup(const ExpertPtrs &ep, bool codes, bool x_f32, const void *x, const float *x_scales, uint32_t W,
                          uint32_t H, uint32_t I, float *hidden, uint32_t *flags, hipStream_t stream)
{
    WideArgs args{};
    args.w0 = ep.gate_w;
    args.w1 = ep.up_w;
    args.s0 = ep.gate_s;
    args.s1 = ep.up_s;
    args.flags = flags;
    args.n_tiles = I / 8;
    args.x = x;
    args.x_scales = x_scales;
    args.W = W;
    args.K = H;
    args.N = I;
    args.y_f32 = hidden;
    const int xt = codes ? WX_CODES : x_f32 ? WX_F32 : WX_BF16;
    const int rt = pick_rt(xt, W, H, args.n_tiles);
    const int t = timer_begin(K_MOE_GATEUP, stream);
    if (codes)
        launch_wide<WK_GATEUP, WX_CODES>(args, rt, stream);
    else if (x_f32)
        launch_wide<WK_GATEUP, WX_F32>(args, rt, stream);
    else
        launch_wide<WK_GATEUP, WX_BF16>(args, rt, stream);
    timer_end(t, stream);
}

uint32_t launch_expert_down(const ExpertPtrs &ep, bool codes, const void *x, const float *x_scales, uint32_t W, uint32_t H,
                            uint32_t I, float *partial, float *out_f32, uint16_t *out_bf16, bool raw, uint32_t *flags,
                            hipStream_t stream)
{
    WideArgs args{};
    args.w0 = ep.down_w;
    args.s0 = ep.down_s;
    args.partial = partial;
    args.flags = flags;
    args.n_tiles = H / 16;
    args.x = x;
    args.x_scales = x_scales;
    args.W = W;
    args.K = I;
    args.N = H;
    args.y_f32 = out_f32;
    args.y_bf16 = out_bf16;
    args.round_f32 = raw ? 0u : 1u;
    args.KS = down_shares(codes, W, I, args.n_tiles);
    const int rt = args.KS > 1 && args.n_tiles > 128 ? 2 : pick_rt(codes ? WX_CODES : WX_F32, W, I, args.n_tiles);
    const int t = timer_begin(K_MOE_DOWN, stream);
    if (codes)
        launch_wide<WK_DOWN, WX_CODES>(args, rt, stream);
    else
        launch_wide<WK_DOWN, WX_F32>(args, rt, stream);
    timer_end(t, stream);
    return args.KS;
}

}  // namespace pw
