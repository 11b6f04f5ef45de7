// The streaming kernel of the block-FP8 projections of 1..32 activation rows (pw_linear.hip) and of
// one expert's forward (pw_expert.hip).
//
// What bounds it: the weights' bytes once, and beside them the activations, which every workgroup
// reads again from L2. A workgroup of 16 weight rows reads W rows of activations for its 16 rows of
// weights: at 13 f32 rows 52 bytes a column (78 as three bf16 planes) against 16. Here a workgroup
// takes 16 RT weight rows over the whole K (pick_rt), its eight waves (launch_wide_16: sixteen) split K,
// and each wave streams its blocks two steps deep with no barrier: the step's activation columns go by
// coalesced direct-to-LDS copies to the wave's own LDS region, the step's weights to registers, and step
// j + 2 is issued as soon as step j is computed. f32 rows are read as f32 and split in registers, once per
// step for all RT tiles. The split sums meet in LDS and are added in split order, so results are
// deterministic.
//
// Measured against one 16-row tile per workgroup with the activations read inside the MFMA loop (us,
// weights in the memory-side cache): 13800 x 4096 (56.5 MB) with 13 f32 rows, mode A, 46.8 -> 15.7
// (3.6 TB/s); 13568 x 4096, mode B with its quantiser launch, 8 f32 rows 19.2 -> 14.7; mode A, f32
// rows, width 1 / 8 / 32 18.7 / 42.2 / 99.4 -> 16.3 / 16.1 / 22.1, bf16 rows 14.5 / 15.4 / 41.8 ->
// 13.7 / 13.7 / 16.5.
#pragma once

#include <type_traits>

#include "pw_device.h"
#include "pw_launch.h"

namespace pw {

template <int XT>
struct WideXBytes {
    static constexpr int value = XT == WX_F32 ? 4 : XT == WX_BF16 ? 2 : 1;
};

constexpr int WAVES = 8;  // of a workgroup (but launch_wide_16's); they split its share of K

// Columns per step: a block, or half a block where two steps of all waves would take more than 128 KB
// of LDS (24 f32 rows and eight waves: 196 KB with whole blocks).
template <int XT, int XR>
struct WideStep {
    static constexpr int value = 128 * WideXBytes<XT>::value * XR * 2 * WAVES <= 131072 ? 128 : 64;
};

// What a workgroup's 16-row tiles are, and what becomes of their sums:
//   WK_PROJ    tiles of a projection's table, K in KS shares of consecutive workgroups; one share: its
//              output rows, rounded or not; more: share sums [KS][W][N].
//   WK_GATEUP  eight gate rows and the same eight up rows of one expert stacked into one tile (output
//              rows 0..7 gate, 8..15 up: lane l takes its gate rows' up values from lane l + 32);
//              SwiGLU -> hidden rows [W][N] f32 (mode B: bf16-staged).
//   WK_DOWN    rows of one expert's down matrix, K in KS shares as above; one share: the output rows
//              rounded, flagged if not finite.
//   WK_BF16    rows of a bf16 weight [N][K] (mode A activations, no scales), K in KS shares as above;
//              the output rows, rounded or not, flagged if not finite.
enum WideKind : int { WK_PROJ = 0, WK_GATEUP = 1, WK_DOWN = 2, WK_BF16 = 3 };

struct WideArgs {
    const ProjTile *tiles;         // WK_PROJ; null: the tensor w0 [N][K]
    const uint8_t *w0, *w1;        // gate and up, down or a projection [N][K], or the bf16 weight's bytes
    const float *s0, *s1;          // ... and their block scales
    float *partial;                // with KS > 1: share sums [KS][W][N]
    uint32_t KS;                   // all but WK_GATEUP
    uint32_t *flags;
    uint32_t n_tiles;
    const void *x;         // activations [W][K]: bf16, f32 or e4m3 codes
    const float *x_scales; // codes: [W][K / 128]
    uint32_t W, K, N;
    float *y_f32;
    uint16_t *y_bf16;
    uint32_t round_f32;
};

// Two f32 -> one dword each of their three bf16 planes, by truncation: every remainder is exact, the
// last has at most eight significant bits, so hi + mid + lo == x as with rounded planes.
__device__ __forceinline__ void split3_pair(float x0, float x1, uint32_t &hi, uint32_t &mid, uint32_t &lo)
{
    const uint32_t b0 = f32_bits(x0), b1 = f32_bits(x1);
    const float r0 = x0 - f32_from(b0 & 0xffff0000u), r1 = x1 - f32_from(b1 & 0xffff0000u);
    const uint32_t c0 = f32_bits(r0), c1 = f32_bits(r1);
    const float s0 = r0 - f32_from(c0 & 0xffff0000u), s1 = r1 - f32_from(c1 & 0xffff0000u);
    hi = __builtin_amdgcn_perm(b1, b0, 0x07060302u);
    mid = __builtin_amdgcn_perm(c1, c0, 0x07060302u);
    lo = __builtin_amdgcn_perm(f32_bits(s1), f32_bits(s0), 0x07060302u);
}

// 16-byte LDS reads of a step slot, waited for in the same block. Written out because the compiler
// cannot tell the two slots apart: ahead of a plain read of one slot it waits for the direct-to-LDS
// copies of the other, and with them for every weight load of the next step (vmcnt 0).
__device__ __forceinline__ uint32_t lds_at(const uint4 *p)
{
    return (uint32_t)(size_t)(const __attribute__((address_space(3))) uint4 *)p;
}
__device__ __forceinline__ void lds_read(const uint32_t (&a)[1], u32x4 (&v)[1])
{
    asm volatile("ds_read_b128 %0, %1\n\ts_waitcnt lgkmcnt(0)" : "=&v"(v[0]) : "v"(a[0]) : "memory");
}
__device__ __forceinline__ void lds_read(const uint32_t (&a)[2], u32x4 (&v)[2])
{
    asm volatile("ds_read_b128 %0, %2\n\tds_read_b128 %1, %3\n\ts_waitcnt lgkmcnt(0)"
                 : "=&v"(v[0]), "=&v"(v[1])
                 : "v"(a[0]), "v"(a[1])
                 : "memory");
}
__device__ __forceinline__ void lds_read(const uint32_t (&a)[4], u32x4 (&v)[4])
{
    asm volatile("ds_read_b128 %0, %4\n\tds_read_b128 %1, %5\n\tds_read_b128 %2, %6\n\tds_read_b128 %3, %7\n\t"
                 "s_waitcnt lgkmcnt(0)"
                 : "=&v"(v[0]), "=&v"(v[1]), "=&v"(v[2]), "=&v"(v[3])
                 : "v"(a[0]), "v"(a[1]), "v"(a[2]), "v"(a[3])
                 : "memory");
}

template <int KIND, int XT, int XR, int RT, int WV>
struct WideStream {
    static constexpr int SC = WideStep<XT, XR>::value;
    static constexpr int XB = WideXBytes<XT>::value;
    static constexpr int NT = (XR + 15) / 16;             // 16-token tiles
    static constexpr int UPR = SC * XB / 16;              // 16-byte units per staged row
    static constexpr int XC = XR * UPR / 64;              // activation copies per step
    static constexpr int WB = KIND == WK_BF16 ? 2 : 1;    // bytes of a weight
    static constexpr int WL = SC * WB / 64;               // weight loads per tile and step
    static constexpr int SLOT = XR * UPR;                 // units per step slot
    static constexpr int RED = WV * RT * NT * 64;         // split partials, in the slots' place
    static constexpr int LDS = 2 * WV * SLOT > RED ? 2 * WV * SLOT : RED;
    static_assert(XR * UPR % 64 == 0, "whole copies");
    static_assert(LDS * 16 <= 160 * 1024, "a workgroup's LDS");

    // Step columns [col, col + SC) of the activation rows -> LDS (row r's unit u at r * UPR + (u ^ (r & 7))):
    // the source of unit c * 64 + lane of the slot.
    static __device__ __forceinline__ const char *x_unit(const char *x, uint32_t W, uint32_t K, uint32_t col, int c,
                                                         int lane)
    {
        const uint32_t p = c * 64 + lane, row = p / UPR, u = (p % UPR) ^ (row & 7);
        const uint32_t r = row < W ? row : W - 1;  // rows past the batch repeat its last row
        return x + ((size_t)r * K + col) * XB + u * 16;
    }

    // the row of tile nt that lane r16 reads (a tile of fewer than sixteen staged rows repeats them)
    static __device__ __forceinline__ uint32_t x_row(int nt, int r16)
    {
        const int rows = XR - nt * 16 < 16 ? XR - nt * 16 : 16;
        return nt * 16 + (r16 & (rows - 1));
    }
};

// AL: the activation rows start on 16 bytes. A step's columns of rows that do not (a caller's slice) go
// through registers while its weights are on their way, so they need no aligned copy in memory (us,
// aligned / off 16 bytes / with a copy launch before it: 13568 x 4096, 8 f32 rows 15.6 / 16.0 / 17.6, 32
// 22.1 / 22.3 / 24.2, 8 bf16 rows 13.7 / 14.2 / 15.8, 32 16.7 / 21.5 / 19.2).
template <int KIND, int XT, int XR, int RT, bool AL = true, int WV = WAVES>
__global__ __launch_bounds__(64 * WV, WV / 4) void wide_kernel(const WideArgs args)
{
    using S = WideStream<KIND, XT, XR, RT, WV>;
    constexpr int NT = S::NT, SC = S::SC, WL = S::WL, XC = S::XC;
    __shared__ uint4 lds_w[S::LDS];  // per wave two step slots; then the split partials [WV][RT * NT][64]
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int q = lane >> 4, r16 = lane & 15;
    const uint32_t K = args.K, W = args.W, blocks = K >> 7;
    const char *x = (const char *)args.x;
    uint4 *slots = lds_w + (size_t)wave * 2 * S::SLOT;

    constexpr int WQ = XT == WX_CODES || KIND == WK_BF16 ? 32 : 16;  // weight bytes of a lane's q in a row
    constexpr bool SHARES = KIND != WK_GATEUP;
    const uint32_t group = SHARES ? blockIdx.x / args.KS : blockIdx.x;
    const uint8_t *wrow[RT];
    const float *ws[RT];
    // One tensor's tiles are formed from the arguments: a descriptor is a trip to memory of its own ahead of
    // the first weight (weights from HBM, us, with / without: 2048 x 4096, one bf16 row 6.1 / 5.75,
    // 13568 x 4096 14.0 / 13.6, one f32 row of 2048 x 4096 6.7 / 6.3).
    if (KIND == WK_PROJ && args.tiles) {
        // the tiles' descriptors in one round trip: all of them are taken before any address is formed
        const uint8_t *wt[RT];
        uint32_t valid[RT];
#pragma unroll
        for (int r = 0; r < RT; ++r) {
            const uint32_t t = group * RT + r;
            const ProjTile *tile = args.tiles + (t < args.n_tiles ? t : args.n_tiles - 1);
            wt[r] = tile->w;
            ws[r] = tile->s;
            valid[r] = tile->valid;
        }
#pragma unroll
        for (int r = 0; r < RT; ++r)
            asm volatile("" ::"s"(wt[r]), "s"(ws[r]), "s"(valid[r]));
#pragma unroll
        for (int r = 0; r < RT; ++r)  // rows past the tile repeat its last row (never stored)
            wrow[r] = wt[r] + (size_t)((uint32_t)r16 < valid[r] ? (uint32_t)r16 : valid[r] - 1) * K + q * WQ;
    } else {
#pragma unroll
        for (int r = 0; r < RT; ++r) {
            const uint32_t t0 = group * RT + r, t = t0 < args.n_tiles ? t0 : args.n_tiles - 1;
            if constexpr (KIND == WK_BF16) {
                const uint32_t row = t * 16 + r16;
                wrow[r] = args.w0 + (size_t)(row < args.N ? row : args.N - 1) * K * 2 + q * WQ;
            } else if constexpr (KIND == WK_GATEUP) {
                wrow[r] = (r16 < 8 ? args.w0 : args.w1) + (size_t)(t * 8 + (r16 & 7)) * K + q * WQ;
                ws[r] = (q < 2 ? args.s0 : args.s1) + (size_t)(t * 8 >> 7) * blocks;
            } else {  // (a projection's last tile may be partial: its rows repeat the last one, never stored)
                const uint32_t row = t * 16 + r16;
                wrow[r] = args.w0 + (size_t)(KIND != WK_PROJ || row < args.N ? row : args.N - 1) * K + q * WQ;
                ws[r] = args.s0 + (size_t)(t * 16 >> 7) * blocks;
            }
        }
    }
    // this wave's blocks (of its workgroup's share of K), and its steps
    uint32_t c0 = 0, cn = blocks;
    if constexpr (SHARES) {
        const uint32_t share = blockIdx.x % args.KS;
        c0 = share * blocks / args.KS;
        cn = (share + 1) * blocks / args.KS - c0;
    }
    const uint32_t b0 = c0 + (uint32_t)wave * cn / WV, b1 = c0 + ((uint32_t)wave + 1) * cn / WV;
    const uint32_t steps = (b1 - b0) * (128 / SC);

    f32x4 total[RT][NT], acc[RT][NT];
#pragma unroll
    for (int r = 0; r < RT; ++r)
#pragma unroll
        for (int nt = 0; nt < NT; ++nt)
            total[r][nt] = acc[r][nt] = f32x4{0.f, 0.f, 0.f, 0.f};

    u32x4 wv[2][RT][WL];
    float sw[2][RT], sa[2][NT];
    // step st into slot s: scales, activation copies, then the weights, in this order in the memory
    // counter (so the youngest XC + RT * WL loads are the copies and weights of the last step issued)
    auto issue = [&](auto s_, uint32_t st) __attribute__((always_inline)) {
        constexpr int s = decltype(s_)::value;
        const uint32_t col = (b0 << 7) + st * SC, b = col >> 7;
        if constexpr (XT == WX_CODES) {
#pragma unroll
            for (int nt = 0; nt < NT; ++nt) {
                const uint32_t row = nt * 16 + r16;
                sa[s][nt] = load_g(args.x_scales + (size_t)(row < W ? row : W - 1) * blocks + b);
            }
        }
        if constexpr (KIND != WK_BF16)
#pragma unroll
            for (int r = 0; r < RT; ++r)
                sw[s][r] = load_g(ws[r] + b);
        asm volatile("" ::: "memory");
        u32x4 xv[AL ? 1 : XC];
#pragma unroll
        for (int c = 0; c < XC; ++c) {
            const char *src = S::x_unit(x, W, K, col, c, lane);
            if constexpr (AL)
                lds_load16(src, slots + s * S::SLOT + c * 64);
            else
                __builtin_memcpy(&xv[c], src, 16);
        }
        asm volatile("" ::: "memory");
#pragma unroll
        for (int r = 0; r < RT; ++r)
#pragma unroll
            for (int h = 0; h < WL; ++h)
                wv[s][r][h] = *(global_u32x4 *)(wrow[r] + (size_t)col * S::WB +
                                                (KIND == WK_BF16 ? (h / 2) * 128 + (h % 2) * 16
                                                                 : h * (XT == WX_CODES ? 16 : 64)));
        asm volatile("" ::: "memory");
        if constexpr (!AL) {  // (the wave's LDS operations keep their order)
#pragma unroll
            for (int c = 0; c < XC; ++c)
                slots[s * S::SLOT + c * 64 + lane] = __builtin_bit_cast(uint4, xv[c]);
            asm volatile("" ::: "memory");
        }
    };
    // N loads issued after step s's own may be outstanding
    auto compute = [&](auto s_, auto n_) __attribute__((always_inline)) {
        constexpr int s = decltype(s_)::value;
        wait_vmcnt<decltype(n_)::value>();
        asm volatile("" ::: "memory");
#pragma unroll
        for (int r = 0; r < RT; ++r)  // the weights' conversions stay behind this wait
#pragma unroll
            for (int h = 0; h < WL; ++h)
                asm volatile("" : "+v"(wv[s][r][h]));
        const uint32_t slot = lds_at(slots + s * S::SLOT);
        if constexpr (XT == WX_CODES) {
#pragma unroll
            for (int nt = 0; nt < NT; ++nt) {
                const uint32_t row = S::x_row(nt, r16), at = slot + row * S::UPR * 16;
                const uint32_t ad[2] = {at + ((q * 2) ^ (row & 7)) * 16, at + ((q * 2 + 1) ^ (row & 7)) * 16};
                u32x4 c[2];
                lds_read(ad, c);
                const i32x8 xb = {(int)c[0][0], (int)c[0][1], (int)c[0][2], (int)c[0][3],
                                  (int)c[1][0], (int)c[1][1], (int)c[1][2], (int)c[1][3]};
#pragma unroll
                for (int r = 0; r < RT; ++r) {
                    const u32x4 w0 = wv[s][r][0], w1 = wv[s][r][WL - 1];
                    const i32x8 wa = {(int)w0[0], (int)w0[1], (int)w0[2], (int)w0[3],
                                      (int)w1[0], (int)w1[1], (int)w1[2], (int)w1[3]};
                    const f32x4 p = mfma_fp8_16x16x128(wa, xb, f32x4{0.f, 0.f, 0.f, 0.f});
#pragma unroll
                    for (int i = 0; i < 4; ++i)
                        total[r][nt][i] = __builtin_fmaf(p[i] * sw[s][r], sa[s][nt], total[r][nt][i]);
                }
            }
        } else {
#pragma unroll
            for (int h = 0; h < SC / 64; ++h) {
                bf16x8 a[RT][2];
#pragma unroll
                for (int r = 0; r < RT; ++r) {
                    if constexpr (KIND == WK_BF16) {
                        a[r][0] = __builtin_bit_cast(bf16x8, wv[s][r][2 * h]);
                        a[r][1] = __builtin_bit_cast(bf16x8, wv[s][r][2 * h + 1]);
                        continue;
                    }
                    a[r][0] = fp8x8_to_bf16x8(wv[s][r][h][0], wv[s][r][h][1]);
                    a[r][1] = fp8x8_to_bf16x8(wv[s][r][h][2], wv[s][r][h][3]);
                }
#pragma unroll
                for (int nt = 0; nt < NT; ++nt) {
                    const uint32_t row = S::x_row(nt, r16), at = slot + row * S::UPR * 16;
                    constexpr int NP = XT == WX_F32 ? 3 : 1;
                    u32x4 pl[NP][2];  // the planes of this lane's sixteen columns
                    if constexpr (XT == WX_BF16) {
                        const uint32_t ad[2] = {at + ((h * 8 + q * 2) ^ (row & 7)) * 16,
                                                at + ((h * 8 + q * 2 + 1) ^ (row & 7)) * 16};
                        lds_read(ad, pl[0]);
                    } else {
                        // Of fewer than sixteen staged rows, each is read by G = 16 / XR lanes of a
                        // DPP row: each splits its share of the sixteen columns, and the first of
                        // them, whose column of the product is the one stored, takes the others' by
                        // row shifts (one row of 1000 x 8192: 11.1 -> 9.8 us).
                        constexpr int G = XR < 16 ? 16 / XR : 1, UG = 4 / G;
                        uint32_t ad[UG];
                        u32x4 u[UG];
#pragma unroll
                        for (int i = 0; i < UG; ++i)
                            ad[i] = at + ((h * 16 + q * 4 + (G > 1 ? (r16 / XR) * UG : 0) + i) ^ (row & 7)) * 16;
                        lds_read(ad, u);
                        uint32_t own[3][2 * UG];
#pragma unroll
                        for (int i = 0; i < 2 * UG; ++i)
                            split3_pair(f32_from(u[i / 2][(i % 2) * 2]), f32_from(u[i / 2][(i % 2) * 2 + 1]), own[0][i],
                                        own[1][i], own[2][i]);
#pragma unroll
                        for (int p = 0; p < NP; ++p)
#pragma unroll
                            for (int i = 0; i < 2 * UG; ++i) {
                                pl[p][i / 4][i % 4] = own[p][i];
                                if constexpr (G >= 2)
                                    pl[p][(2 * UG + i) / 4][(2 * UG + i) % 4] = dpp_u32<0x100 + XR % 16, 0xf>(own[p][i]);
                                if constexpr (G == 4) {
                                    pl[p][1][i % 4] = dpp_u32<0x100 + 2 * XR % 16, 0xf>(own[p][i]);
                                    pl[p][1][(2 + i) % 4] = dpp_u32<0x100 + 3 * XR % 16, 0xf>(own[p][i]);
                                }
                            }
                    }
#pragma unroll
                    for (int p = 0; p < NP; ++p) {
                        const bf16x8 x0 = __builtin_bit_cast(bf16x8, pl[p][0]), x1 = __builtin_bit_cast(bf16x8, pl[p][1]);
#pragma unroll
                        for (int r = 0; r < RT; ++r) {
                            acc[r][nt] = mfma_bf16_16x16x32(a[r][0], x0, acc[r][nt]);
                            acc[r][nt] = mfma_bf16_16x16x32(a[r][1], x1, acc[r][nt]);
                        }
                    }
                }
            }
            // A block is complete. Blocks are added to the total also where no scale asks for it: a
            // wave's whole share of K in one accumulator is a chain of 1024 columns at K = 8192, whose
            // error against 64 bits is 3.6e-7 (f32 rows) and 1.9e-7 (bf16 rows) where block sums have
            // 1.6e-7 and 1.0e-7, at the same speed.
            if constexpr (SC == 128 || s == 1) {
#pragma unroll
                for (int r = 0; r < RT; ++r)
#pragma unroll
                    for (int nt = 0; nt < NT; ++nt) {
#pragma unroll
                        for (int i = 0; i < 4; ++i) {
                            if constexpr (KIND == WK_BF16)
                                total[r][nt][i] += acc[r][nt][i];
                            else
                                total[r][nt][i] = __builtin_fmaf(sw[s][r], acc[r][nt][i], total[r][nt][i]);
                        }
                        acc[r][nt] = f32x4{0.f, 0.f, 0.f, 0.f};
                    }
            }
        }
        asm volatile("" ::: "memory");  // the slot's reads stay ahead of its next copies
    };
    // two steps in flight; no issue inside a condition, so the wait for one step's weights never
    // has to assume that the next step's were not issued
    using I0 = std::integral_constant<int, 0>;
    using I1 = std::integral_constant<int, 1>;
    using Next = std::integral_constant<int, XC + RT * WL>;
    if (steps >= 2) {
        issue(I0{}, 0);
        issue(I1{}, 1);
        uint32_t st = 0;
        for (; st + 4 <= steps; st += 2) {
            compute(I0{}, Next{});
            issue(I0{}, st + 2);
            compute(I1{}, Next{});
            issue(I1{}, st + 3);
        }
        compute(I0{}, Next{});
        if (SC == 128 && st + 3 == steps) {
            issue(I0{}, st + 2);
            compute(I1{}, Next{});
            compute(I0{}, I0{});
        } else {
            compute(I1{}, I0{});
        }
    } else if (steps == 1) {
        issue(I0{}, 0);
        compute(I0{}, I0{});
    }

    // the split partials in LDS over the slots (every wave is past its reads), summed in split order
    __syncthreads();
    f32x4 *red = (f32x4 *)lds_w;
#pragma unroll
    for (int r = 0; r < RT; ++r)
#pragma unroll
        for (int nt = 0; nt < NT; ++nt)
            red[(wave * RT * NT + r * NT + nt) * 64 + lane] = total[r][nt];
    __syncthreads();
    if (wave >= RT * NT)
        return;
    const uint32_t t = group * RT + wave / NT, token = (wave % NT) * 16 + r16;
    if (t >= args.n_tiles)
        return;
    f32x4 sum = red[wave * 64 + lane];
#pragma unroll
    for (int w = 1; w < WV; ++w) {
        const f32x4 o = red[(w * RT * NT + wave) * 64 + lane];
#pragma unroll
        for (int i = 0; i < 4; ++i)
            sum[i] += o[i];
    }
    if constexpr (KIND == WK_PROJ) {
        if (token >= W)
            return;
        const uint32_t out_row = args.tiles ? args.tiles[t].out_row : t * 16;
        const uint32_t valid = args.tiles ? args.tiles[t].valid : args.N - t * 16;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const uint32_t row = q * 4 + i;
            if (row >= valid)
                continue;
            const size_t at = (size_t)token * args.N + out_row + row;
            if (args.KS > 1) {
                args.partial[(size_t)(blockIdx.x % args.KS) * W * args.N + at] = sum[i];
                continue;
            }
            if (args.y_f32)
                args.y_f32[at] = args.round_f32 ? round_bf16(sum[i]) : sum[i];
            if (args.y_bf16)
                args.y_bf16[at] = bf16_bits(sum[i]);
        }
    } else if constexpr (KIND == WK_GATEUP) {
        float up[4];
#pragma unroll
        for (int i = 0; i < 4; ++i)
            up[i] = __shfl(sum[i], (lane + 32) & 63, 64);
        if (token >= W || q >= 2)
            return;
        bool bad = false;
        float o[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            if constexpr (XT == WX_CODES) {  // bf16_staged_swiglu
                const float gv = round_bf16(sum[i]), uv = round_bf16(up[i]);
                o[i] = round_bf16(silu_bf16_staged(gv) * uv);
                bad |= !finite_f32(gv) || !finite_f32(uv) || !finite_f32(o[i]);
            } else {
                o[i] = (sum[i] / (1.0f + expf(-sum[i]))) * up[i];
                bad |= !finite_f32(o[i]);
            }
        }
        *(float4 *)(args.y_f32 + (size_t)token * args.N + t * 8 + q * 4) = make_float4(o[0], o[1], o[2], o[3]);
        if (bad)
            raise_flag(args.flags, FLAG_SWIGLU_NONFINITE);
    } else if constexpr (KIND == WK_BF16) {
        if (token >= W)
            return;
        bool bad = false;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const uint32_t row = t * 16 + q * 4 + i;
            if (row >= args.N)
                continue;
            const size_t at = (size_t)token * args.N + row;
            if (args.KS > 1) {
                args.partial[(size_t)(blockIdx.x % args.KS) * W * args.N + at] = sum[i];
                continue;
            }
            const float r = round_bf16(sum[i]);
            bad |= !finite_f32(r);
            if (args.y_f32)
                args.y_f32[at] = args.round_f32 ? r : sum[i];
            if (args.y_bf16)
                args.y_bf16[at] = (uint16_t)(f32_bits(r) >> 16);
        }
        if (bad)
            raise_flag(args.flags, FLAG_ROUND_NONFINITE);
    } else {
        if (token >= W)
            return;
        const size_t at = (size_t)token * args.N + t * 16 + q * 4;
        if (args.KS > 1) {
            float *p = args.partial + (size_t)(blockIdx.x % args.KS) * W * args.N + at;
            *(float4 *)p = make_float4(sum[0], sum[1], sum[2], sum[3]);
            return;
        }
        bool bad = false;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const float r = round_bf16(sum[i]);
            bad |= !finite_f32(r);
            if (args.y_f32)
                args.y_f32[at + i] = args.round_f32 ? r : sum[i];
            if (args.y_bf16)
                args.y_bf16[at + i] = (uint16_t)(f32_bits(r) >> 16);
        }
        if (bad)
            raise_flag(args.flags, FLAG_ROUND_NONFINITE);
    }
}

// Tiles per workgroup. One generation of workgroups over the 256 CUs reads the activations least and
// has no second start: one tile up to 256 tiles, two up to 512, then four. Where a row's activations
// are few bytes beside the weights, several small workgroups per CU beat half a chip of larger ones, and
// keep more loads in flight where the weights come from HBM: up to four rows of bf16 or codes take one
// tile, but from 769 to 1024 tiles three and four rows two, and of 6144 columns and more four; eight
// rows one from 513 to 768 (us, K = 4096, one / two / four tiles, weights in the memory-side cache |
// from HBM: bf16 width 1, 938 tiles 13.1 / 12.8 / 12.3 | 14.3 / 14.4 / 16.5, 1024 tiles
// 13.3 / 13.4 / 13.0 | 14.7 / 15.2 / 17.9; width 4, 848 tiles 12.5 / 12.3 / 12.0 | 14.4 / 14.2 / 15.5; of
// 8192 columns, 769 tiles, width 4 19.9 / 21.5 / 19.1 | 22.5 / 24.4 / 22.7; f32 width 16, 257 tiles
// 14.8 / 11.2 / 15.4, 512 tiles 17.4 / 12.2 / 16.8, 532 tiles 23.5 / 20.4 / 16.7). Past 1024 tiles
// four tiles are several generations of one workgroup per CU, each with its own start: up to eight rows
// take one tile, batches of up to 32 activation bytes a column two (us of a whole 4096 x 16384 expert,
// 2048 gate/up tiles: bf16 width 1 40.9 / 44.2 / 47.8, width 16 52.2 / 50.2 / 53.7, width 32
// 86.2 / 76.4 / 70.8; codes width 24 66.2 / 58.4 / 59.1).
// Up to 2048 columns a wave has one or two steps, all in flight at once, so more tiles a workgroup
// give it nothing to overlap: smaller workgroups keep ahead for longer (us, one / two / four tiles:
// width 8, 1024 tiles of 1024 columns 6.8 / 6.4 / 6.8; f32 width 1, 532 tiles of 1024 columns
// 6.9 / 6.5 / 7.1, of 2048 9.4 / 9.1 / 9.7).
static inline int pick_rt(int xt, uint32_t W, uint32_t K, uint32_t n_tiles)
{
    const bool light = xt != WX_F32 && W <= 4, medium = xt != WX_F32 && W <= 8;
    if (light && (n_tiles <= 256 || n_tiles > 1024))
        return 1;
    if (light && n_tiles > 768)
        return K <= 2048 ? 1 : K >= 6144 ? 4 : W <= 2 ? 1 : 2;
    if (K <= 2048 && n_tiles > 512 && n_tiles <= 1024 && (medium ? n_tiles > 768 : xt == WX_F32 && W <= 4 && n_tiles <= 768))
        return 2;
    if (n_tiles > 1024)
        return medium ? 1 : W * (xt == WX_F32 ? 4 : xt == WX_BF16 ? 2 : 1) <= 32 ? 2 : 4;
    if (light || n_tiles <= 256 || (medium && n_tiles > 512 && n_tiles <= 768))
        return 1;
    return n_tiles <= 512 ? 2 : 4;
}

template <int KIND>
static dim3 wide_grid(const WideArgs &args, int rt)
{
    return dim3((args.n_tiles + rt - 1) / (uint32_t)rt * (KIND != WK_GATEUP ? args.KS : 1u));
}

template <int KIND, int XT, int XR>
static void launch_wide_rt(const WideArgs &args, int rt, hipStream_t stream)
{
    const dim3 grid = wide_grid<KIND>(args, rt), block(512);
    if (rt == 4)
        hipLaunchKernelGGL((wide_kernel<KIND, XT, XR, 4>), grid, block, 0, stream, args);
    else if (KIND == WK_BF16 && rt == 3)
        hipLaunchKernelGGL((wide_kernel<KIND, XT, XR, KIND == WK_BF16 ? 3 : 2>), grid, block, 0, stream, args);
    else if (rt == 2)
        hipLaunchKernelGGL((wide_kernel<KIND, XT, XR, 2>), grid, block, 0, stream, args);
    else
        hipLaunchKernelGGL((wide_kernel<KIND, XT, XR, 1>), grid, block, 0, stream, args);
}

// Staged rows: the batch's, rounded up to 4 (not for codes, whose eight rows are one copy), 8, 16,
// 24 (f32) or 32.
template <int KIND, int XT>
static void launch_wide(const WideArgs &args, int rt, hipStream_t stream)
{
    if (XT != WX_CODES && args.W <= 4)
        launch_wide_rt<KIND, XT, XT != WX_CODES ? 4 : 8>(args, rt, stream);
    else if (args.W <= 8)
        launch_wide_rt<KIND, XT, 8>(args, rt, stream);
    else if (args.W <= 16)
        launch_wide_rt<KIND, XT, 16>(args, rt, stream);
    else if (XT == WX_F32 && args.W <= 24)
        launch_wide_rt<KIND, XT, XT == WX_F32 ? 24 : 32>(args, rt, stream);
    else
        launch_wide_rt<KIND, XT, 32>(args, rt, stream);
}

// One tile of up to four rows on sixteen waves.
template <int KIND, bool AL>
static void launch_wide_16(int xt, const WideArgs &args, hipStream_t stream)
{
    const dim3 grid = wide_grid<KIND>(args, 1), block(1024);
    if (xt == WX_F32)
        hipLaunchKernelGGL((wide_kernel<KIND, WX_F32, 4, 1, AL, 16>), grid, block, 0, stream, args);
    else
        hipLaunchKernelGGL((wide_kernel<KIND, WX_BF16, 4, 1, AL, 16>), grid, block, 0, stream, args);
}

// Rows off 16 bytes: eight, sixteen or 32 staged rows, one or four tiles.
template <int KIND, int XT, int XR>
static void launch_unaligned_xr(const WideArgs &args, int rt, hipStream_t stream)
{
    const dim3 grid = wide_grid<KIND>(args, rt), block(512);
    if (rt == 1)
        hipLaunchKernelGGL((wide_kernel<KIND, XT, XR, 1, false>), grid, block, 0, stream, args);
    else
        hipLaunchKernelGGL((wide_kernel<KIND, XT, XR, 4, false>), grid, block, 0, stream, args);
}

template <int KIND, int XT>
static void launch_wide_unaligned(const WideArgs &args, int rt, hipStream_t stream)
{
    rt = rt == 1 ? 1 : 4;
    if (args.W <= 8)
        launch_unaligned_xr<KIND, XT, 8>(args, rt, stream);
    else if (args.W <= 16)
        launch_unaligned_xr<KIND, XT, 16>(args, rt, stream);
    else
        launch_unaligned_xr<KIND, XT, 32>(args, rt, stream);
}

}  // namespace pw
