// Depthwise 3x3 (stride 1 or 2) + the pointwise 1x1 convolution that consumes it as ONE kernel: a block owns TH x TW pixels of
// one image over all channels between the layers, and 16 NW CG of the output channels.
//
//   * The halo of the tile, all channels, is requested at once (one round trip), with the constants of both layers, and lies in
//     LDS as [channels / 16][halo pixel][16 bytes]: the depthwise operands are 16-byte reads of neighbouring pixels, and an odd
//     number of pieces per channel group keeps the staging writes on different banks.
//   * Depthwise: v_mfma_i32_16x16x64_i8 with pixels as rows and channels as columns, the weights of a tap diagonal (a column keeps
//     one byte of the 16).  A wave takes 64 channels as four groups: tap slots 0 .. 3 and 4 .. 7 are one operand read per group,
//     the ninth taps of the four groups share a third (lane group g reads group g, and only that group's weights are not zero).
//     A lane then holds one channel of four pixels in each group, so its constants are one 16-byte row entry for four groups;
//     four channels per lane, as DepthwiseMfmaKernel has them, took five reads per group and made LDS bandwidth the bound (14 x
//     14 x 512, one image 6.0 -> 5.5 us).  Its four codes of a pixel -- channels j, 16 + j, 32 + j, 48 + j -- are one dword, which
//     goes back to LDS over the halo just read; the pointwise weights are packed with their channels in that order.
//   * Pointwise: a wave owns 16 CG output channels of all pixels and reads its weights in operand order straight from L2 (runs of
//     1 KB; 55 bytes a clock and CU were measured for that, 14 to 20 for 128-byte rows through LDS with a wait per k-tile), the
//     first k-steps requested ahead of the depthwise phase.  No barrier inside: two after the halo, two around the write-out.
//   * The outputs meet in LDS and leave as 16 bytes per lane.
// At many tiles VALU work is the largest share, most of it the requantization of both layers: 14 x 14 x 512, 64 images, with 25
// instructions and a branch per four values 12 k of a SIMD's 27 k cycles issued VALU and 5.6 k matrix instructions; the rest of a
// wave's life is waits, at barriers and for the weights (82 MB through the CUs' L1s).  (Now 23 instructions, fewer of them
// conversions, and a branch per 16 values: a pass of MobileNetV1 at 64 images 177.3 -> 170.2 us, most of it here.)  At few tiles
// it is the chain of round trips.  Times against the kernel with a k-tile loop it replaces (64 images | 256): 14 x 14 x 512 -> 512
// 15.4 -> 12.8 | 54.2 -> 35.7 us, 28 x 28 x 256 -> 256 20.2 -> 17.7 | 68.9 -> 61.3, 28 x 28 x 256 -> 14 x 14 x 512 11.2 -> 10.7 | 43.1 ->
// 34.8; against two launches, one image | eight: 14 x 14 x 512 7.6 -> 5.5 | 9.3 -> 7.5, 28 x 28 x 256 7.2 -> 4.6 | 8.6 -> 6.3.
// Both layers' arithmetic is untouched -- exact int32 sums, the same requantization routine with the same constants -- so the
// bytes are those of the two layers run one after the other.
#pragma once

#include <hip/hip_runtime.h>

#include "common.h"
#include "conv_kernels.h"
#include "device_math.h"
#include "dw_mfma_kernel.h"

namespace mi355x
{

struct DwPwPanelArgs
{
    // depthwise 3x3, multiplier 1, C % 16 == 0
    const uint8_t*  x;
    const uint8_t*  pad16;      // 16 bytes that become the depthwise padding value under dw_xor
    const uint32_t* dw_blk;     // constants per block of 64 channels: kDwBlkRows rows of [16][4] dwords
    int H, W, C, Ho, Wo;
    int pad_top, pad_left;
    int tiles_x, tiles_y, nb;   // nb: blocks per tile (output channels / (16 NW CG), rounded up)
    int total_items, xcd_chunk;
    uint32_t rcp_tiles_x, rcp_tiles_y, rcp_nb, rcp_ng;      // ceil(2^32 / d) of tiles_x, tiles_y, nb and C / 16
    uint32_t dw_xor;
    Requant dw_rq;
    // pointwise 1x1 over C channels
    const int8_t*  w;           // operand order (PackFragKernel)
    int            co_groups;   // groups of 16 channels w holds
    ChanTab        pw_ct;
    const int32_t* pw_corr;
    uint8_t*       y;
    long long      y_bytes;
    int            Co;
    int            zw_neg;      // AW: minus the zero point of the weights
    uint32_t       mid_xor;     // 0x80808080 when the tensor between the layers is uint8: the panel holds the int8-shifted codes
    Requant        pw_rq;
};

// what accumulators start from, m, b, mult, biasf, filter taps 0 .. 3, 4 .. 7, 8, and those of the second halves
constexpr int kDwBlkRows = 11;

template <int S, int TH, int TW, int NW, int CG>
struct DwPwPanelGeom
{
    static_assert(TW == 4 || TW == 8 || TW == 16, "a group of 16 pixels is whole tile rows");
    static constexpr int NT = 64 * NW;
    static constexpr int PX = TH * TW, PG = PX / 16;
    static constexpr int HR = (TH - 1) * S + 3, HC = (TW - 1) * S + 3, HPX = HR * HC;
    static constexpr int GP = (HPX | 1) * 16;            // bytes per group of 16 channels in LDS: an odd number of 16-byte pieces
    static constexpr int NCOL = 16 * NW * CG;            // output channels of a block
    static constexpr int OP = NCOL + 16;                 // bytes per pixel of the output staging
    static constexpr int Panel(int C)                    // halo and panel, later the output staging
    {
        const int in = (C + 63) / 64 * 4 * GP, out = PX * OP;
        return in > out ? in : out;
    }
    // behind it the depthwise layer's constants and five rows of NCOL dwords of the pointwise layer's
    static constexpr int TB(bool u) { return (u ? kDwBlkRows : kDwBlkRows - 3) * 256; }        // bytes per 64 channels
    static constexpr int Smem(int C, bool u) { return Panel(C) + (C + 63) / 64 * TB(u) + 20 * NCOL; }
};

// KS: k-steps of 64 channels where the instance fixes them (64 (KS - 1) < C <= 64 KS), 0: a.C decides.  U: depthwise weights in two
// halves, pointwise weights with a zero point.
template <int S, int TH, int TW, int NW, int CG, int KS, bool U>
__global__ __launch_bounds__(64 * NW, 4) void DwPwPanelKernel(DwPwPanelArgs a)
{
    using G = DwPwPanelGeom<S, TH, TW, NW, CG>;
    constexpr int NT = G::NT, PG = G::PG, HC = G::HC, HPX = G::HPX, GP = G::GP, OP = G::OP;
    constexpr int RPG = 16 / TW;                         // tile rows per group of 16 pixels
    constexpr int DEPTH = CG >= 4 ? 2 : CG == 2 ? 4 : 8;
    constexpr int RD = KS != 0 && KS < DEPTH ? KS : DEPTH;   // k-steps of weights in flight
    constexpr int HS = KS != 0 ? (HPX * KS * 4 + NT - 1) / NT : 6;   // halo pieces of a thread in flight
    // depthwise work: blocks of 64 channels go to the waves in turn, all PG groups of 16 pixels of a block to one wave (UC at a
    // time); with fewer blocks than waves, WPB waves share a block
    constexpr int WPB = KS != 0 && NW / KS >= 2 ? (NW / KS < PG ? NW / KS : PG) : 1;
    constexpr int UW = PG / WPB, UC = WPB > 1 ? UW : UW < 2 || U ? 1 : 2;
    static_assert(PG % WPB == 0 && UW % UC == 0, "whole shares");
    // Pixel groups requantized together.  (With U the registers are full: batches of 2 and 4 spill, 57.4 against 56.4 us for a pass of
    // 13 images at width 0.75.)
    constexpr int PB = U ? 1 : PG < 4 ? PG : 4;
    constexpr bool EARLY = PG == 1 || (PG == 2 && !U);                      // registers for weights requested ahead of the depthwise phase
    constexpr int TB = G::TB(U);
    constexpr int TS = KS != 0 ? (KS * (TB / 16) + G::NCOL / 4 * 5 + NT - 1) / NT : 4;      // ... and table pieces
    extern __shared__ __attribute__((aligned(16))) uint8_t panel_lds[];   // [C / 16][GP]: halo pixels, then panel pixels, of 16 bytes

    int b = XcdContiguousWorkItem(blockIdx.x, a.xcd_chunk);
    if ((static_cast<int>(blockIdx.x) >> 3) >= a.xcd_chunk || b >= a.total_items) return;
    int q = DivByInvariant(b, a.nb, a.rcp_nb);
    const int bn = b - q * a.nb; b = q;
    q = DivByInvariant(b, a.tiles_x, a.rcp_tiles_x);
    const int tx = b - q * a.tiles_x; b = q;
    const int n = DivByInvariant(b, a.tiles_y, a.rcp_tiles_y);
    const int ty = b - n * a.tiles_y;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int j = lane & 15, g = lane >> 4;
    const int ng = a.C >> 4;                             // groups of 16 channels between the layers
    const int steps = KS != 0 ? KS : (a.C + 63) >> 6;

    // ---- weights of the wave's CG groups of output channels ---------------------------------------------------------------------
    v4i wv[RD][CG];
    auto load_weights = [&](int ks, int r) {
#pragma unroll
        for (int c = 0; c < CG; ++c)
            wv[r][c] = *reinterpret_cast<const v4i*>(a.w + static_cast<long long>(min((bn * NW + wave) * CG + c, a.co_groups - 1) * steps + ks) * 1024 + lane * 16);
    };
    // ---- tables ---------------------------------------------------------------------------------------------------------------------
    uint8_t* const tab = panel_lds + G::Panel(64 * steps);
    uint8_t* const ptab = tab + steps * TB;
    const int dw_pieces = steps * (TB / 16), tab_pieces = dw_pieces + G::NCOL / 4 * 5;
    auto tab_src = [&](int i) -> const void* {
        if (i < dw_pieces)
        {
            const int blk = i / (TB / 16);
            return a.dw_blk + blk * (kDwBlkRows * 64) + (i - blk * (TB / 16)) * 4;
        }
        i -= dw_pieces;
        const int r = i / (G::NCOL / 4), c4 = min(bn * G::NCOL + (i - r * (G::NCOL / 4)) * 4, a.co_groups * 16 - 4);
        if (r == 2) return a.pw_corr + c4;
        return a.pw_ct.p + (r < 2 ? r + 2 : r - 3) * a.pw_ct.stride + c4;        // m, b, ., mult, biasf
    };

    // ---- the halo of the tile, all channels ---------------------------------------------------------------------------------------
    {
        const int iy_org = ty * TH * S - a.pad_top, ix_org = tx * TW * S - a.pad_left;
        const uint8_t* const xn = a.x + static_cast<long long>(n) * a.H * a.W * a.C;
        const int xm = static_cast<int>(a.dw_xor);
        const int pieces = HPX * ng;
        for (int i0 = 0; KS != 0 ? i0 == 0 : i0 < pieces; i0 += NT * HS)
        {
            v4i h[HS];
            int at[HS];
#pragma unroll
            for (int k = 0; k < HS; ++k)
            {
                at[k] = -1;
                if (i0 + k * NT >= pieces) continue;
                const int i = min(i0 + k * NT + tid, pieces - 1);
                const int px = DivByInvariant(i, ng, a.rcp_ng);
                const int part = i - px * ng;
                const int row = px / HC, col = px - row * HC;
                const int iy = iy_org + row, ix = ix_org + col;
                const bool ok = static_cast<unsigned>(iy) < static_cast<unsigned>(a.H) && static_cast<unsigned>(ix) < static_cast<unsigned>(a.W);
                h[k] = *reinterpret_cast<const v4i*>(ok ? xn + (iy * a.W + ix) * a.C + part * 16 : a.pad16);
                if (i0 + k * NT + tid < pieces) at[k] = part * GP + px * 16;
            }
            if (i0 == 0)
            {
                v4i t[TS];
#pragma unroll
                for (int k = 0; k < TS; ++k)
                    if (KS != 0 || k * NT < tab_pieces) t[k] = *reinterpret_cast<const v4i*>(tab_src(min(tid + k * NT, tab_pieces - 1)));
                if constexpr (EARLY)
                {
#pragma unroll
                    for (int r = 0; r < RD; ++r)
                        if (r < steps) load_weights(r, r);
                }
#pragma unroll
                for (int k = 0; k < TS; ++k)
                    if (tid + k * NT < tab_pieces) *reinterpret_cast<v4i*>(tab + (tid + k * NT) * 16) = t[k];
            }
#pragma unroll
            for (int k = 0; k < HS; ++k)
                if (at[k] >= 0) *reinterpret_cast<v4i*>(panel_lds + at[k]) = h[k] ^ xm;
        }
        if (KS == 0)
            for (int i = tid + TS * NT; i < tab_pieces; i += NT) *reinterpret_cast<v4i*>(tab + i * 16) = *reinterpret_cast<const v4i*>(tab_src(i));
    }
    __syncthreads();

    // ---- depthwise: a wave takes 64 channels and writes their codes over the halo it has just read ------------------------------
    {
        const int rj = j / TW, cj = j % TW;
        int dtap[3];
#pragma unroll
        for (int m = 0; m < 3; ++m)
        {
            const int t = m < 2 ? 4 * m + g : 8;
            dtap[m] = ((rj * S + t / 3) * HC + cj * S + t % 3) * 16;
        }
        // weight operand: byte j of the lane's 16 is byte b of `taps`, the others are zero
        uint32_t sel[4], sel8[4];
#pragma unroll
        for (int d = 0; d < 4; ++d)
        {
            sel[d] = (j >> 2) == d ? 0x0c0c0c0cu ^ (static_cast<uint32_t>(0x0c ^ g) << (8 * (j & 3))) : 0x0c0c0c0cu;
            sel8[d] = (j >> 2) == d ? 0x0c0c0c0cu ^ (0x0cu << (8 * (j & 3))) : 0x0c0c0c0cu;
        }
        auto operand = [&](uint32_t taps, const uint32_t (&s)[4]) {
            v4i o;
#pragma unroll
            for (int d = 0; d < 4; ++d) o[d] = static_cast<int>(__builtin_amdgcn_perm(0u, taps, s[d]));
            return o;
        };
        // exact sums of UC pixel groups from u0 on, channel 64 blk + 16 e + j of pixels 4 g .. 4 g + 3 in acc[e]
        auto sums = [&](int blk, int u0, v4i (&acc)[4][UC]) {
            const uint8_t* const tb = tab + blk * TB + j * 16;
            const uint8_t* const hu = panel_lds + blk * (4 * GP) + u0 * (RPG * S * HC * 16);
            const v4i corr = *reinterpret_cast<const v4i*>(tb);
            v4i w[3], w2[3];
#pragma unroll
            for (int m = 0; m < 3; ++m)
            {
                w[m] = *reinterpret_cast<const v4i*>(tb + (5 + m) * 256);
                if constexpr (U) w2[m] = *reinterpret_cast<const v4i*>(tb + (8 + m) * 256);
            }
            // the ninth tap of the four channel groups shares one operand: lane group g reads it from channel group g
            v4i x8[UC];
#pragma unroll
            for (int u = 0; u < UC; ++u) x8[u] = *reinterpret_cast<const v4i*>(hu + g * GP + dtap[2] + u * (RPG * S * HC * 16));
#pragma unroll
            for (int e = 0; e < 4; ++e)
            {
                const v4i w03 = operand(w[0][e], sel), w47 = operand(w[1][e], sel), w8 = operand(g == e ? w[2][e] : 0, sel8);
                v4i v03, v47, v8;
                if constexpr (U) { v03 = operand(w2[0][e], sel); v47 = operand(w2[1][e], sel); v8 = operand(g == e ? w2[2][e] : 0, sel8); }
#pragma unroll
                for (int u = 0; u < UC; ++u)
                {
                    const v4i x0 = *reinterpret_cast<const v4i*>(hu + e * GP + dtap[0] + u * (RPG * S * HC * 16));
                    const v4i x1 = *reinterpret_cast<const v4i*>(hu + e * GP + dtap[1] + u * (RPG * S * HC * 16));
                    v4i v = v4i{corr[e], corr[e], corr[e], corr[e]};
                    v = __builtin_amdgcn_mfma_i32_16x16x64_i8(x0, w03, v, 0, 0, 0);
                    v = __builtin_amdgcn_mfma_i32_16x16x64_i8(x1, w47, v, 0, 0, 0);
                    v = __builtin_amdgcn_mfma_i32_16x16x64_i8(x8[u], w8, v, 0, 0, 0);
                    if constexpr (U)
                    {
                        v = __builtin_amdgcn_mfma_i32_16x16x64_i8(x0, v03, v, 0, 0, 0);
                        v = __builtin_amdgcn_mfma_i32_16x16x64_i8(x1, v47, v, 0, 0, 0);
                        v = __builtin_amdgcn_mfma_i32_16x16x64_i8(x8[u], v8, v, 0, 0, 0);
                    }
                    acc[e][u] = v;
                }
            }
        };
        auto codes = [&](int blk, int u0, const v4i (&acc)[4][UC]) {
            const uint8_t* const tb = tab + blk * TB + j * 16;
            const Fast4 f[1] = {{*reinterpret_cast<const float4*>(tb + 256), *reinterpret_cast<const float4*>(tb + 512)}};
            uint8_t* const out = panel_lds + blk * (4 * GP) + (j >> 2) * GP + (16 * u0 + 4 * g) * 16 + (j & 3) * 4;
#pragma unroll
            for (int u = 0; u < UC; ++u)
            {
                v4i v[4];
                uint32_t q[4];
#pragma unroll
                for (int r = 0; r < 4; ++r) v[r] = v4i{acc[0][u][r], acc[1][u][r], acc[2][u][r], acc[3][u][r]};
                RequantCore<true, 4, 1>(v, q, f, a.dw_rq, [&](int, float4& m, float4& b) {
                    m = *reinterpret_cast<const float4*>(tb + 768);
                    b = *reinterpret_cast<const float4*>(tb + 1024);
                });
#pragma unroll
                for (int r = 0; r < 4; ++r) *reinterpret_cast<uint32_t*>(out + (16 * u + r) * 16) = q[r] ^ a.mid_xor;
            }
        };
        if constexpr (WPB > 1)
        {
            const int blk = wave / WPB, u0 = wave % WPB * UW;
            v4i acc[4][UC];
            if (blk < KS) sums(blk, u0, acc);
            __syncthreads();                             // all have read the halo
            if (blk < KS) codes(blk, u0, acc);
        }
        else
        {
            // A pixel group's codes go to pixels 16 u .. 16 u + 15 of the block, and the later groups read halo pixels from
            // (u + 1) RPG S HC on, behind them: a wave may write before it reads on.
            static_assert(RPG * S * HC >= 16, "a later pixel group reads behind what an earlier one writes");
            for (int blk = wave; blk < steps; blk += NW)
#pragma unroll
                for (int u0 = 0; u0 < UW; u0 += UC)
                {
                    v4i acc[4][UC];
                    sums(blk, u0, acc);
                    codes(blk, u0, acc);
                }
        }
        if constexpr (!EARLY)
        {
#pragma unroll
            for (int r = 0; r < RD; ++r)
                if (r < steps) load_weights(r, r);
        }
    }
    __syncthreads();

    // ---- pointwise ------------------------------------------------------------------------------------------------------------------
    v4i acc[CG][PG];
    int xs[PG];
#pragma unroll
    for (int p = 0; p < PG; ++p)
    {
        xs[p] = 0;
#pragma unroll
        for (int c = 0; c < CG; ++c) acc[c][p] = *reinterpret_cast<const v4i*>(ptab + (2 * G::NCOL + (wave * CG + c) * 16 + 4 * g) * 4);
    }
    const uint8_t* const pb = panel_lds + g * GP + j * 16;
    // The sum of a pixel's codes is over the channels that exist.  Those that complete the last block of 64 hold whatever the
    // activation between the layers makes of them (their weights are zero, so the products do not mind); they are the high bytes
    // of each dword of the last k-step.
    const int last_ones = static_cast<int>(0x01010101u >> (8 * (-ng & 3)));
    for (int k0 = 0; k0 < steps; k0 += RD)
    {
#pragma unroll
        for (int r = 0; r < RD; ++r)
        {
            const int ks = k0 + r;
            if (ks >= steps) break;
            v4i xb[PG];
#pragma unroll
            for (int p = 0; p < PG; ++p) xb[p] = *reinterpret_cast<const v4i*>(pb + ks * 4 * GP + p * 256);
#pragma unroll
            for (int c = 0; c < CG; ++c)
#pragma unroll
                for (int p = 0; p < PG; ++p) acc[c][p] = __builtin_amdgcn_mfma_i32_16x16x64_i8(wv[r][c], xb[p], acc[c][p], 0, 0, 0);
            if constexpr (U)
            {
                const int ones = ks == steps - 1 ? last_ones : 0x01010101;
#pragma unroll
                for (int p = 0; p < PG; ++p)
#pragma unroll
                    for (int d = 0; d < 4; ++d) xs[p] = __builtin_amdgcn_sdot4(xb[p][d], ones, xs[p], false);
            }
            if (ks + RD < steps) load_weights(ks + RD, r);
        }
    }

    // ---- write-out --------------------------------------------------------------------------------------------------------------------
    if constexpr (U)
    {
#pragma unroll
        for (int p = 0; p < PG; ++p)
        {
            xs[p] += __shfl_xor(xs[p], 16);
            xs[p] += __shfl_xor(xs[p], 32);
            xs[p] *= a.zw_neg;
        }
    }
    __syncthreads();                                     // the panel has been read; the outputs take its place
    WithBits(a.pw_rq, [&](auto bits) {
#pragma unroll
    for (int c = 0; c < CG; ++c)
    {
        const uint8_t* const tc = ptab + ((wave * CG + c) * 16 + 4 * g) * 4;
        const Fast4 f = {*reinterpret_cast<const float4*>(tc), *reinterpret_cast<const float4*>(tc + 4 * G::NCOL)};
        const ChanTab exact{reinterpret_cast<const float*>(tc) + 3 * G::NCOL, G::NCOL};
#pragma unroll
        for (int p0 = 0; p0 < PG; p0 += PB)
        {
            v4i v[PB];
            uint32_t out[PB];
#pragma unroll
            for (int i = 0; i < PB; ++i)
            {
                v[i] = acc[c][p0 + i];
                if constexpr (U) v[i] += xs[p0 + i];
            }
            RequantPixels<decltype(bits)::value, PB>(v, out, f, exact, 0, a.pw_rq);
#pragma unroll
            for (int i = 0; i < PB; ++i) *reinterpret_cast<uint32_t*>(panel_lds + (16 * (p0 + i) + j) * OP + (wave * CG + c) * 16 + 4 * g) = out[i];
        }
    }
    });
    __syncthreads();
    const OutPtr outp = MakeOutPtr(a.y, a.y_bytes);
    constexpr int CHUNKS = NW * CG;                      // 16-byte pieces per pixel
    constexpr int NP = (G::PX * CHUNKS + NT - 1) / NT;
#pragma unroll
    for (int i = 0; i < NP; ++i)
    {
        const int idx = tid + i * NT;
        const int r = idx / CHUNKS, chunk = idx - r * CHUNKS;
        const int oy = ty * TH + r / TW, ox = tx * TW + r % TW, c0 = bn * G::NCOL + chunk * 16;
        if (r < G::PX && oy < a.Ho && ox < a.Wo && c0 < a.Co)
            StoreOut16(outp, ((static_cast<long long>(n) * a.Ho + oy) * a.Wo + ox) * a.Co + c0, *reinterpret_cast<const v4i*>(panel_lds + r * OP + chunk * 16));
    }
}

} // namespace mi355x
