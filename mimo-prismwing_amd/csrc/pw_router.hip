// Routed-MoE router on the device: logits, PyTorch sigmoid, noaux-tc top-8 and renormalised
// weights, so the routes a layer consumes never leave HBM (route_mlp, src/text_endpoint.rs:
// 4342-4380; Metal router GEMV kernels/block_fp8_gemv.metal:317-356).
//
// Logits use this build's declared summation order: a workgroup of 256 threads takes one expert;
// thread g accumulates x[c] * w[e, c] with a fused multiply-add over the 8-column groups
// c0 = 8g, 8g + 2048, 8g + 4096, ... (columns c0 .. c0 + 7 in order), each wave of 64 partials is
// reduced by a halving tree (lane l += lane l + offset, offset 32 .. 1) into w0..w3, and the logit
// is (w0 + w1) + (w2 + w3). The reference's order belongs to Apple Accelerate's SGEMM, which is
// closed; any fixed order is within the routes' tolerance of it, and this one is restated by the
// oracle so the device routes can be checked bit for bit. Scores are the PyTorch sigmoid on the
// SLEEF expf_u10 restatement; the selection and weights are pytorch_noaux_routes (pw_topk.h), with
// nth_element run on the row held in one wave's registers (pw_select_wave.h: the same result, the
// same partition order).
#include "pw_device.h"
#include "pw_launch.h"
#include "pw_select_wave.h"

namespace pw {

// Eight consecutive values of a row: bf16 (one 16-byte load) or f32 (two), loaded raw and
// widened to f32 by unpack.
template <typename T>
struct Raw8;
template <>
struct Raw8<uint16_t> {
    uint4 q;
    __device__ __forceinline__ void load(const uint16_t *p) { q = load_global16(p); }
    __device__ __forceinline__ void unpack(float *v) const
    {
        const uint32_t u[4] = {q.x, q.y, q.z, q.w};
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            v[2 * i] = f32_from(u[i] << 16);
            v[2 * i + 1] = f32_from(u[i] & 0xffff0000u);
        }
    }
};
template <>
struct Raw8<float> {
    uint4 q0, q1;
    __device__ __forceinline__ void load(const float *p)
    {
        q0 = load_global16(p);
        q1 = load_global16(p + 4);
    }
    __device__ __forceinline__ void unpack(float *v) const
    {
        const uint32_t u[8] = {q0.x, q0.y, q0.z, q0.w, q1.x, q1.y, q1.z, q1.w};
#pragma unroll
        for (int i = 0; i < 8; ++i)
            v[i] = f32_from(u[i]);
    }
};

// v + (the value of lane l + OFF) at lanes l < OFF <= 8 (a row_shl DPP move: both lanes in the
// lane's 16-lane row; the other lanes get values of no use)
template <int OFF>
__device__ __forceinline__ float add_from_lane_above(float v)
{
    return v + __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x100 + OFF,
                                                                     0xf, 0xf, false));
}

// One workgroup per (expert, chunk of up to 8 rows; NR rows loaded, NR >= the chunk's rows):
// scores[p][e] = sigmoid(logit[p][e]) in the declared order. Every thread reads its 8-column
// groups of the expert row and of the chunk's rows with 16-byte loads (rows past the chunk's last
// reread that row, so every load is in bounds and none waits on a branch: a thread's loads of two
// column groups go out together); the activation rows are shared by all experts' workgroups
// through L2. The halving trees of the NR rows run interleaved, their steps within 16 lanes as
// DPP moves.
template <typename TX, typename TW, int NR>
__global__ __launch_bounds__(256) void router_scores_kernel(const TX *__restrict__ x, const TW *__restrict__ w,
                                                            uint32_t rows, uint32_t E, uint32_t K,
                                                            float *__restrict__ scores)
{
    __shared__ float wave_sum[NR][4];
    const uint32_t g = threadIdx.x, lane = g & 63, wave = g >> 6;
    const uint32_t e = blockIdx.x;
    const uint32_t p0 = blockIdx.y * 8;
    const uint32_t np = rows - p0 < (uint32_t)NR ? rows - p0 : (uint32_t)NR;
    float acc[NR];
    const TX *xr[NR];
#pragma unroll
    for (int j = 0; j < NR; ++j) {
        acc[j] = 0.0f;
        xr[j] = x + (size_t)(p0 + ((uint32_t)j < np ? (uint32_t)j : np - 1)) * K;
    }
    const TW *wrow = w + (size_t)e * K;
    // column groups c0 = 8 g + 2048 i in ascending i, two per pass
    for (uint32_t c0 = 8 * g; c0 < K; c0 += 4096) {
        const bool has1 = c0 + 2048 < K;
        const uint32_t c1 = has1 ? c0 + 2048 : c0;
        Raw8<TW> w0, w1;
        Raw8<TX> x0[NR], x1[NR];
        w0.load(wrow + c0);
        w1.load(wrow + c1);
#pragma unroll
        for (int j = 0; j < NR; ++j) {
            x0[j].load(xr[j] + c0);
            x1[j].load(xr[j] + c1);
        }
        // every load above is issued before the first use below
        __builtin_amdgcn_sched_barrier(0);
        float wv[8], xv[8];
        w0.unpack(wv);
#pragma unroll
        for (int j = 0; j < NR; ++j) {
            x0[j].unpack(xv);
#pragma unroll
            for (int c = 0; c < 8; ++c)
                acc[j] = __builtin_fmaf(xv[c], wv[c], acc[j]);
        }
        // the second group's sums are kept only where it exists (computed anyway, so its loads
        // stay with the first group's)
        w1.unpack(wv);
#pragma unroll
        for (int j = 0; j < NR; ++j) {
            x1[j].unpack(xv);
            float t = acc[j];
#pragma unroll
            for (int c = 0; c < 8; ++c)
                t = __builtin_fmaf(xv[c], wv[c], t);
            acc[j] = has1 ? t : acc[j];
        }
    }
    // each wave's halving tree (lane l += lane l + off, off = 32 .. 1), ending in lane 0
#pragma unroll
    for (int j = 0; j < NR; ++j)
        acc[j] = acc[j] + __shfl_down(acc[j], 32, 64);
#pragma unroll
    for (int j = 0; j < NR; ++j)
        acc[j] = acc[j] + __shfl_down(acc[j], 16, 64);
#pragma unroll
    for (int j = 0; j < NR; ++j) {
        acc[j] = add_from_lane_above<8>(acc[j]);
        acc[j] = add_from_lane_above<4>(acc[j]);
        acc[j] = add_from_lane_above<2>(acc[j]);
        acc[j] = add_from_lane_above<1>(acc[j]);
    }
    if (lane == 0) {
#pragma unroll
        for (int j = 0; j < NR; ++j)
            wave_sum[j][wave] = acc[j];
    }
    __syncthreads();
    if (g < np) {
        const float logit = (wave_sum[g][0] + wave_sum[g][1]) + (wave_sum[g][2] + wave_sum[g][3]);
        scores[(size_t)(p0 + g) * E + e] = sigmoid_pytorch(logit);
    }
}

// The same scores for many rows, in the same declared order, as a contraction on the matrix cores:
// v_mfma_f32_16x16x1 multiplies 16 rows by 16 experts for one column of each of four column groups
// and adds the products to four separate accumulators, each with the rounding of one fused
// multiply-add, so a chain of sixteen of them at hidden 4096 is the partial sums of four column groups
// of every (row, expert) of the tile. Bound: the kernel above re-reads eight rows per expert from L2
// (4.7 GB at 2048 rows x 256 experts, 270 us); a 16 x 16 tile reads an eighth of that, and runs within
// about twice the matrix cores' time for the 2.1 G products (27 us).
//
// Work item: 16 rows x 16 experts. Wave v takes the column groups g = 64 v .. 64 v + 63 (its quarter of
// the declared order) in quads: groups l, l + 1, l + 2, l + 3 of each of the four runs l + {0, 32, 16,
// 48}, run r in the MFMA's block r, so the first two levels of the halving tree (offsets 32 and 16) are
// sums of a lane's own accumulators, and the later ones (8, 4, 2, 1) are sums of earlier quads'
// results that the lane still holds. A quad's columns of one 2048-column pass (64 contiguous bf16
// bytes per row and run) go straight from global memory into the wave's own LDS, the next step's
// while this step's are multiplied (no barrier before the end); their 16-byte units are XOR-swizzled
// by row, so the operand reads (16 rows of one unit) spread over the banks.
template <typename T>
struct RsTile {
    static constexpr uint32_t EPU = 16 / sizeof(T);       // values per 16-byte unit
    static constexpr uint32_t U = 4 * 8 / EPU;            // units of a quad's 32 columns, per row and run
    static constexpr uint32_t UNITS = 4 * 16 * U;         // units of a step: four runs, 16 rows
    static constexpr uint32_t RPC = 64 / U, CPR = 16 / RPC; // rows per 64-lane copy, copies per run
    static constexpr uint32_t JU = U / 4;                 // units of one group's eight columns
    __device__ __forceinline__ static uint32_t swizzle(uint32_t row) { return U == 4 ? (row >> 1) & 3 : row & 7; }
    // the lane's source offsets (values) within the tile's rows; rows past the last reread it
    __device__ __forceinline__ static void offsets(uint32_t (&off)[CPR], uint32_t row0, uint32_t n_rows, uint32_t K,
                                                   uint32_t lane)
    {
#pragma unroll
        for (uint32_t c = 0; c < CPR; ++c) {
            const uint32_t r = RPC * c + lane / U, left = n_rows - 1 - row0;
            off[c] = (r < left ? r : left) * K + ((lane % U) ^ swizzle(r)) * EPU;
        }
    }
    // a step's columns of the tile's rows (src: the first row at the step's first column) -> LDS
    // [run][row][unit]
    __device__ __forceinline__ static void copy(const T *src, const uint32_t (&off)[CPR], uint4 *lds)
    {
#pragma unroll
        for (uint32_t run = 0; run < 4; ++run)
#pragma unroll
            for (uint32_t c = 0; c < CPR; ++c)
                lds_load16(src + off[c] + 8 * (run == 1 ? 32 : run == 2 ? 16 : run == 3 ? 48 : 0),
                           lds + (run * CPR + c) * 64);
    }
    // the units of this lane's row (lane % 16) and run (lane / 16) for group j of the quad
    __device__ __forceinline__ static void read(const uint4 *lds, uint32_t lane, uint32_t j, uint4 (&q)[JU])
    {
        const uint32_t r = lane & 15;
#pragma unroll
        for (uint32_t i = 0; i < JU; ++i)
            q[i] = lds[lane * U + ((JU * j + i) ^ swizzle(r))];
    }
    __device__ __forceinline__ static float value(const uint4 (&q)[JU], int c)
    {
        const uint4 &u = q[c / EPU];
        if constexpr (JU == 1) {
            const uint32_t d[4] = {u.x, u.y, u.z, u.w};
            return f32_from(c & 1 ? d[c >> 1] & 0xffff0000u : d[c >> 1] << 16);
        } else {
            const uint32_t d[4] = {u.x, u.y, u.z, u.w};
            return f32_from(d[c & 3]);
        }
    }
};

template <typename TX, typename TW>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(sizeof(TX) + sizeof(TW) == 4 ? 3 : 2))) void router_scores_tile_kernel(const TX *__restrict__ x, const TW *__restrict__ w,
                                                                 uint32_t rows, uint32_t E, uint32_t K,
                                                                 float *__restrict__ scores)
{
    using X = RsTile<TX>;
    using W = RsTile<TW>;
    constexpr uint32_t STEP = X::UNITS + W::UNITS;  // 16-byte units of one step
    extern __shared__ uint4 lds_rs[];               // per wave one step; then [4][256] wave sums
    const uint32_t tid = threadIdx.x, lane = tid & 63;
    const uint32_t wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(tid >> 6));
    const uint32_t n_et = (E + 15) >> 4, n_rt = (rows + 15) >> 4;
    // workgroup i runs on XCD i % 8: with eight row tiles or more, an XCD takes whole row tiles, so
    // each L2 holds the router's weights and its own rows (fewer: row tiles over all XCDs)
    uint32_t rt, et;
    if (n_rt >= 8) {
        const uint32_t j = blockIdx.x >> 3;
        rt = (blockIdx.x & 7) + 8 * (j / n_et);
        et = j % n_et;
    } else {
        rt = blockIdx.x / n_et;
        et = blockIdx.x % n_et;
    }
    if (rt >= n_rt)
        return;
    uint4 *buf = lds_rs + wave * STEP;
    const uint32_t passes = K >> 11;
    uint32_t xo[X::CPR], wo[W::CPR];
    X::offsets(xo, rt * 16, rows, K, lane);
    W::offsets(wo, et * 16, E, K, lane);
    const TX *xb = x + (size_t)rt * 16 * K + 512 * wave;
    const TW *wb = w + (size_t)et * 16 * K + 512 * wave;
    X::copy(xb, xo, buf);
    W::copy(wb, wo, buf + X::UNITS);
    // the halving tree after offsets 32 and 16, group l = 4 quad + j of the sixteen: offset 8 adds
    // quad 2 to quad 0 and quad 3 to quad 1 (the order they run in), offset 4 the second sum to the
    // first, offsets 2 and 1 groups within the quad
    f32x4 part[2][4];
#pragma unroll
    for (uint32_t k = 0; k < 4; ++k) {
        const uint32_t quad = 2 * (k & 1) + (k >> 1), next = 2 * ((k + 1) & 1) + ((k + 1) >> 1);
        f32x16 acc[4];
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
            for (int i = 0; i < 16; ++i)
                acc[j][i] = 0.0f;
        uint32_t p = 0;
#pragma unroll 1
        do {
            // the step's columns are in LDS; its operands into registers, then the next step's copies
            // overwrite the buffer while this step is multiplied
            wait_vmcnt<0>();
            asm volatile("" ::: "memory");
            uint4 xq[4][X::JU], wq[4][W::JU];
#pragma unroll
            for (uint32_t j = 0; j < 4; ++j) {
                X::read(buf, lane, j, xq[j]);
                W::read(buf + X::UNITS, lane, j, wq[j]);
            }
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
            const bool last = p + 1 == passes;
            if (k < 3 || !last) {
                const uint32_t col = last ? 32 * next : 32 * quad + 2048 * (p + 1);
                X::copy(xb + col, xo, buf);
                W::copy(wb + col, wo, buf + X::UNITS);
            }
#pragma unroll
            for (int c = 0; c < 8; ++c) {
#pragma unroll
                for (uint32_t j = 0; j < 4; ++j)
                    acc[j] = __builtin_amdgcn_mfma_f32_16x16x1f32(X::value(xq[j], c), W::value(wq[j], c), acc[j], 0, 0,
                                                                  0);
                __builtin_amdgcn_sched_barrier(0);  // the widened values stay a column at a time
            }
        } while (++p < passes);  // K is a positive multiple of 2048
        // lane: rows 4 (lane / 16) + i, expert lane % 16; acc[j][4 r + i]: run r (offsets 0, 32, 16, 48)
#pragma unroll
        for (uint32_t j = 0; j < 4; ++j)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const float v = (acc[j][i] + acc[j][4 + i]) + (acc[j][8 + i] + acc[j][12 + i]);
                part[k >> 1][j][i] = (k & 1) == 0 ? v : part[k >> 1][j][i] + v;
            }
        // formed here: left to itself the compiler keeps all four quads' accumulators (in scratch
        // memory) and adds them at the end
#pragma unroll
        for (uint32_t j = 0; j < 4; ++j)
            asm volatile("" : "+v"(part[k >> 1][j]));
    }
    f32x4 sum;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        float t[4];
#pragma unroll
        for (int j = 0; j < 4; ++j)
            t[j] = part[0][j][i] + part[1][j][i];
        sum[i] = (t[0] + t[2]) + (t[1] + t[3]);
    }
    __syncthreads();  // every wave is done with its steps
    float *sums = (float *)lds_rs;
#pragma unroll
    for (int i = 0; i < 4; ++i)
        sums[wave * 256 + (4 * (lane >> 4) + i) * 16 + (lane & 15)] = sum[i];
    __syncthreads();
    const uint32_t row = rt * 16 + (tid >> 4), e = et * 16 + (tid & 15);
    if (row < rows && e < E) {
        const float logit = (sums[tid] + sums[256 + tid]) + (sums[512 + tid] + sums[768 + tid]);
        scores[(size_t)row * E + e] = sigmoid_pytorch(logit);
    }
}

// One wave per row: the row's corrected scores stay in the wave's registers (position p = 64 c +
// lane in register c), select_route_row runs the top-8 partition on them (pw_select_wave.h), and
// lane 0 writes the row. A row that fails (non-finite score or bias, a broken top-k, invalid
// weights) raises FLAG_ROUTE and gets expert ids E (which the layer schedule rejects) with zero
// weights.
template <int NC>
__global__ __launch_bounds__(64) void router_select_kernel(const float *__restrict__ scores,
                                                           const float *__restrict__ bias, uint32_t rows,
                                                           uint32_t E, uint32_t *__restrict__ selected,
                                                           float *__restrict__ weights, uint32_t *tie_rows,
                                                           uint32_t *flags)
{
    __shared__ TopkEntry lds_pairs[64 * NC];
    const uint32_t p = blockIdx.x;
    if (p >= rows)
        return;
    DeviceWave w;
    uint32_t sel_k;
    float w_k;
    bool tie = false;
    const int st = select_route_row<NC>(w, scores + (size_t)p * E, bias, E, lds_pairs, sel_k, w_k, &tie);
    const uint32_t lane = w.lane();
    if (st != ROUTE_OK) {
        sel_k = E;
        w_k = 0.0f;
        tie = false;
        if (lane == 0)
            raise_flag(flags, FLAG_ROUTE);
    }
    if (lane < 8) {
        selected[(size_t)p * 8 + lane] = sel_k;
        weights[(size_t)p * 8 + lane] = w_k;
    }
    if (lane == 0 && tie && tie_rows)
        atomicAdd(tie_rows, 1u);
}

// The tile kernel runs from this many 16 x 16 tiles on (half the CUs): a tile is a chain of 16 to 32
// memory round trips (about 15 us at hidden 4096), which fewer tiles do not repay. Scores and
// selection, us, row kernel / tile kernel: 100 rows x 256 experts 30.8 / 31.1, 128 rows 33.9 / 30.7,
// 2048 rows 209.5 / 75.6; hidden 2048, 64 experts: 200 rows 18.6 / 17.9, 512 rows 23.9 / 20.4.
constexpr uint32_t ROUTER_TILES = 128;

template <typename TX, typename TW>
static void launch_scores_xw(const TX *x, const TW *w, uint32_t rows, uint32_t E, uint32_t K, float *scores,
                             hipStream_t stream)
{
    const uint32_t n_et = (E + 15) / 16, n_rt = (rows + 15) / 16;
    if (K % 2048 == 0 && n_et * n_rt >= ROUTER_TILES) {
        const uint32_t tiles = n_rt >= 8 ? 8 * ((n_rt + 7) / 8) * n_et : n_rt * n_et;
        constexpr size_t lds = (size_t)4 * (RsTile<TX>::UNITS + RsTile<TW>::UNITS) * 16;
        static_assert(lds <= 65536, "the default LDS limit");
        hipLaunchKernelGGL((router_scores_tile_kernel<TX, TW>), dim3(tiles), dim3(256), lds, stream, x, w, rows, E, K,
                           scores);
        return;
    }
    const dim3 grid(E, (rows + 7) / 8), block(256);
    if (rows == 1) hipLaunchKernelGGL((router_scores_kernel<TX, TW, 1>), grid, block, 0, stream, x, w, rows, E, K, scores);
    else if (rows == 2) hipLaunchKernelGGL((router_scores_kernel<TX, TW, 2>), grid, block, 0, stream, x, w, rows, E, K, scores);
    else if (rows <= 4) hipLaunchKernelGGL((router_scores_kernel<TX, TW, 4>), grid, block, 0, stream, x, w, rows, E, K, scores);
    else hipLaunchKernelGGL((router_scores_kernel<TX, TW, 8>), grid, block, 0, stream, x, w, rows, E, K, scores);
}

template <typename TX>
static void launch_scores_x(const TX *x, const void *w, bool w_f32, uint32_t rows, uint32_t E, uint32_t K,
                            float *scores, hipStream_t stream)
{
    if (w_f32)
        launch_scores_xw(x, (const float *)w, rows, E, K, scores, stream);
    else
        launch_scores_xw(x, (const uint16_t *)w, rows, E, K, scores, stream);
}

void launch_router_scores(const void *x, bool x_f32, const void *w, bool w_f32, uint32_t rows, uint32_t E,
                          uint32_t K, float *scores, hipStream_t stream)
{
    if (x_f32)
        launch_scores_x<float>((const float *)x, w, w_f32, rows, E, K, scores, stream);
    else
        launch_scores_x<uint16_t>((const uint16_t *)x, w, w_f32, rows, E, K, scores, stream);
}

void launch_router_select(const float *scores, const float *bias, uint32_t rows, uint32_t E, uint32_t *selected,
                          float *weights, uint32_t *tie_rows, uint32_t *flags, hipStream_t stream)
{
#define PW_SELECT(NC)                                                                                         \
    hipLaunchKernelGGL(router_select_kernel<NC>, dim3(rows), dim3(64), 0, stream, scores, bias, rows, E, selected, \
                       weights, tie_rows, flags)
    if (E <= 64) PW_SELECT(1);
    else if (E <= 128) PW_SELECT(2);
    else if (E <= 256) PW_SELECT(4);
    else if (E <= 512) PW_SELECT(8);
    else PW_SELECT(16);
#undef PW_SELECT
}

void launch_router(const void *x, bool x_f32, const void *w, bool w_f32, const float *bias, uint32_t rows,
                   uint32_t E, uint32_t K, float *scores, uint32_t *selected, float *weights, uint32_t *tie_rows,
                   uint32_t *flags, hipStream_t stream)
{
    const int t = timer_begin(K_ROUTER, stream);
    launch_router_scores(x, x_f32, w, w_f32, rows, E, K, scores, stream);
    launch_router_select(scores, bias, rows, E, selected, weights, tie_rows, flags, stream);
    timer_end(t, stream);
}

}  // namespace pw
