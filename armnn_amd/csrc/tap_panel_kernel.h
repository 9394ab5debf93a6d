// Convolutions with filters of more than one tap, and some 1x1 layers: a block owns BM consecutive output pixels x BN output channels.
//
//   * Output pixels of a launch are numbered through rows and images, input pixels likewise, so that the input pixels any tap of the
//     block's outputs reads lie between the first tap of its first and the last tap of its last one (tap_panel_run.h): one contiguous run
//     of memory, which goes to LDS whole, as [channels / 16][pixel][16 bytes], in one round trip.  A tap is then an offset into it; what falls
//     into the padding (the run has other rows' pixels there) reads 16 prepared bytes instead, by one bit per tap and pixel.
//   * Weights come in operand order straight from L2 (runs of 1 KB), RD k-steps ahead: no staging, no barrier inside the products.
//   * KG waves share an output tile and split K, the others lie side by side over channels and pixels.  The partial tiles meet in LDS; each
//     wave adds up and requantizes its share.
// What these launches take is not matrix instructions but what a wave does around them, one instruction after the other, cold from the
// instruction cache.  Cycle stamps at 14 x 14 x 256, 16 images, 64 x 64 tiles over four waves of K (196 blocks), first form -> now: arguments and requests
// of weights 2.2 k -> 1.6 k, pixels and their taps 3.5 k -> 0.6 k (one pixel per lane and a shuffle, no loops), requests of the panel 1.8 k -> 0.6 k
// (its bytes are contiguous), the panel's arrival 1.6 k, partial tiles 1.4 k, requantization 1.3 k, stores 0.5 k; the products, 6.7 k for 2.3 k of matrix
// instructions, took the launch from 7.1 to 6.3 us when a tap's select moved out of its k-steps and pointers only counted.  Weights
// that lie in L1 (one k-step read again and again), deeper rings of them (6 and 9 k-steps) and pixel operands read a k-step ahead changed nothing.
// Before -> here, from graphs, three sets of tensors in turn: 3 x 3, 16 images, 28 x 28 x 128 7.7 -> 6.4 us, 14 x 14 x 256 8.7 -> 6.5, 7 x 7 x 512 13.6 -> 6.4, 14 x
// 14 x 512 at stride 2 13.7 -> 8.7; 64 images, 14 x 14 x 256 18.3 -> 12.8, 28 x 28 x 128 15.6 -> 12.7; 40 x 40 x 192, 32 images, 43.8 -> 23.8; 20 x 20 x 432 -> 75, 20
// images, 29.8 -> 9.1; 5 x 5 over 28 x 28 x 64 -> 256, 16 images, 15.8 -> 10; one image, 14 x 14 x 256 5.26 -> 4.40, 7 x 7 x 512 7.26 -> 5.40.  ResNet-50, three
// networks in turn: one image 112.8 -> 99.5 us a pass (3.9 of it the 28 x 28 x 128 -> 512 layers, which have one tap), 32 images 403.6 -> 375.
#pragma once

#include <hip/hip_runtime.h>

#include "common.h"
#include "conv_kernels.h"
#include "device_math.h"
#include "dw_mfma_kernel.h"
#include "tap_panel_run.h"

namespace mi355x
{

struct TapPanelArgs
{
    IgemmArgs g;                    // g.w in operand order; tiles_n = ceil(Co / columns of a block), tiles_m = ceil(M / pixels of a block)
    int gp;                         // bytes per 16 channels of the panel: an odd number of 16-byte pieces, the last one padding
    int in_pixels;                  // batch * H * W
    int panel_bytes;                // of all channels
    uint32_t tap_rows;              // bits 0, Kw, 2 Kw, ... (Kh - 1) Kw
    uint32_t rcp_pr, rcp_minor;     // ceil(2^32 / d) of the 16-byte pieces per pixel and of minor
    uint32_t rcp_dy, rcp_dx;        // ... and of the dilations
    struct { int step, ky, kx, ci; } wave_k[5];     // where each share of K starts: k-step, and the filter tap and byte of it that begins there
    int minor, by_columns;          // the faster index of a tile is its row, of tiles_m, or its column, of tiles_n
};

// Waves over pixels, channels and K; a wave's groups of 16 channels and of 16 pixels.
template <int WM, int WN, int WK, int CG, int PG>
struct TapPanelGeom
{
    static constexpr int NW = WM * WN * WK, NCOL = 16 * CG * WN, PX = 16 * PG * WM, OP = NCOL + 16;
    // what one of the WK waves finishes: PO groups of pixels, of which CO groups of channels
    static constexpr int PO = PG >= WK ? PG / WK : 1, CO = PG >= WK ? CG : CG * PG / WK;
    static_assert(PG >= WK ? PG % WK == 0 : WK % PG == 0 && CG * PG % WK == 0, "whole shares");
    static constexpr int FirstP(int wk) { return PG >= WK ? wk * PO : wk * PG / WK; }
    static constexpr int FirstC(int wk) { return PG >= WK ? 0 : wk % (WK / PG) * CO; }
    static constexpr int kPartial = WK > 1 ? WM * WN * WK * (WK - 1) * PO * CO * 1024 : 0;
    static constexpr int Work(int panel)
    {
        const int out = PX * OP;
        const int w = panel > out ? panel : out;
        return w > kPartial ? w : kPartial;
    }
    static constexpr int Smem(int panel) { return Work(panel) + 20 * NCOL; }        // + m, b, mult, biasf, corr of the block's channels
};

// The tiles: K split over KG waves, BM pixels x BN channels of a block; waves over pixels and channels, a wave's groups of 16 channels and pixels,
// k-steps of weights in flight.
template <int KG, int BM, int BN>
struct TapTile
{
    static constexpr int WM = BM == 128 ? 2 : KG == 1 ? 2 : 1;
    static constexpr int CG = BM == 128 && KG == 2 ? 4 : 2;
    static constexpr int WN = BN / (16 * CG), PG = BM / (16 * WM), RD = CG == 4 ? 3 : 4;
    static constexpr int WAVES = WM * WN * KG, WAVES_PER_SIMD = CG == 4 ? 3 : 4;
    using Geom = TapPanelGeom<WM, WN, KG, CG, PG>;
    static_assert(Geom::NCOL == BN && Geom::PX == BM, "the tile");
};

// AW: the weights have a zero point (row sums beside the products).  RG: Ci is no multiple of 16 (g.Ck bytes per pixel in LDS).  WHOLE: Ci is a
// multiple of 64, a filter tap whole k-steps.
template <int WM, int WN, int WK, int CG, int PG, int RD, bool AW, bool RG, bool WHOLE>
__device__ __forceinline__ void TapPanelBlock(const TapPanelArgs& t)
{
    using G = TapPanelGeom<WM, WN, WK, CG, PG>;
    static_assert(!(RG && WHOLE), "channels that are no multiple of 16 make no whole k-steps");
    constexpr int NW = G::NW, NT = 64 * NW, NCOL = G::NCOL, PX = G::PX, PO = G::PO, CO = G::CO, OP = G::OP, HS = NW == 4 ? 6 : 4;
    extern __shared__ __attribute__((aligned(16))) uint8_t tap_lds[];
    FetchArgs<sizeof(TapPanelArgs)>();
    const IgemmArgs& a = t.g;
    const int nblocks = a.tiles_m * a.tiles_n, per_xcd = (nblocks + 7) >> 3;
    const int tile = XcdContiguousWorkItem(blockIdx.x, per_xcd);
    if (static_cast<int>(blockIdx.x >> 3) >= per_xcd || tile >= nblocks) return;
    const int major = DivByInvariant(tile, t.minor, t.rcp_minor), minor = tile - major * t.minor;
    const int tm = t.by_columns ? minor : major, tn = t.by_columns ? major : minor;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wk = wave / (WM * WN), wm = wave / WN % WM, wn = wave % WN;
    const int j = lane & 15, g = lane >> 4;
    const int xm = static_cast<int>(a.xor_mask);
    const int tap_bytes = RG ? a.Ck : a.Ci;

    // ---- weights of the wave's CG groups of output channels, its part of K ---------------------------------------------------------------
    const int steps = (a.Kh * a.Kw * tap_bytes + 63) >> 6;
    const int s0 = t.wave_k[wk].step, s1 = t.wave_k[wk + 1].step;
    const int8_t* wp[CG];
#pragma unroll
    for (int c = 0; c < CG; ++c) wp[c] = a.w + (static_cast<long long>(tn * (NCOL / 16) + wn * CG + c) * steps + s0) * 1024;
    uint32_t w_at = static_cast<uint32_t>(lane * 16);    // of the next k-step to be requested
    v4i wv[RD][CG];
    auto load_weights = [&](int r) {
#pragma unroll
        for (int c = 0; c < CG; ++c) wv[r][c] = *reinterpret_cast<const v4i*>(wp[c] + w_at);
        w_at += 1024;
    };
#pragma unroll
    for (int r = 0; r < RD; ++r)
        if (s0 + r < s1) load_weights(r);

    // ---- output pixel `lane` of each 64 of the wave's: its first tap's number, and which taps lie inside the image ---------------------------------------
    constexpr int EV = (PG + 3) / 4, WPX = 16 * PG;
    int first[EV];
    uint32_t taps[EV];
#pragma unroll
    for (int e = 0; e < EV; ++e)
    {
        const int m = min(tm * PX + wm * WPX + e * 64 + (WPX < 64 ? lane & (WPX - 1) : lane), a.M - 1);     // pixels past the end repeat the last one (never stored)
        const int r = DivByInvariant(m, a.Wo, a.wo_magic);
        const int n = DivByInvariant(r, a.Ho, a.ho_magic);
        const int iy = (r - n * a.Ho) * a.stride_y - a.pad_top, ix = (m - r * a.Wo) * a.stride_x - a.pad_left;
        first[e] = (n * a.H + iy) * a.W + ix;
        const auto itself = [](int v) { return v; };
        taps[e] = a.dil_x == 1 && a.dil_y == 1
                      ? TapsInside(iy, ix, a.H, a.W, a.Kh, a.Kw, 1, 1, t.tap_rows, itself, itself)
                      : TapsInside(iy, ix, a.H, a.W, a.Kh, a.Kw, a.dil_y, a.dil_x, t.tap_rows, [&](int v) { return DivByInvariant(v, a.dil_y, t.rcp_dy); },
                                   [&](int v) { return DivByInvariant(v, a.dil_x, t.rcp_dx); });
    }
    // first taps of the block's first and last pixel
    int base, last;
    if constexpr (WM == 1)
    {
        base = __builtin_amdgcn_readfirstlane(first[0]);
        last = __builtin_amdgcn_readlane(first[EV - 1], WPX < 64 ? WPX - 1 : 63);
    }
    else
    {
        const auto first_of = [&](int m) {
            const int r = DivByInvariant(m, a.Wo, a.wo_magic), n = DivByInvariant(r, a.Ho, a.ho_magic);
            return (n * a.H + (r - n * a.Ho) * a.stride_y - a.pad_top) * a.W + (m - r * a.Wo) * a.stride_x - a.pad_left;
        };
        base = first_of(tm * PX);
        last = first_of(min(tm * PX + PX, a.M) - 1);
    }
    const int npx = last - base + (a.Kh - 1) * a.dil_y * a.W + (a.Kw - 1) * a.dil_x + 1;

    // ---- the input pixels base .. base + npx - 1, all channels ------------------------------------------------------------------------
    const int pr = tap_bytes >> 4, pieces = npx * pr;
    const int lo = max(0, -base) * pr, hi = min(npx, t.in_pixels - base) * pr - 1;       // pieces inside the tensor
    const uint8_t* const run = a.x + static_cast<long long>(base) * a.Ci;
    const int sh = 31 - __clz(pr);
    const bool pow2 = (pr & (pr - 1)) == 0;
    v4i h[HS];
    int back[RG ? HS : 1];
    auto load_panel = [&](int i0) {
#pragma unroll
        for (int k = 0; k < HS; ++k)
        {
            if (i0 + k * NT >= pieces) continue;
            const int i = PieceInside(i0 + k * NT + tid, lo, hi);
            if constexpr (RG)
            {
                const int px = DivByInvariant(i, pr, t.rcp_pr);
                const uint8_t* src = run + (px * a.Ci + (i - px * pr) * 16);
                back[k] = src > a.x_last16 ? static_cast<int>(src - a.x_last16) : 0;
                h[k] = LoadUnaligned16(src - back[k]);
            }
            else h[k] = *reinterpret_cast<const v4i*>(run + i * 16);
        }
    };
    auto store_panel = [&](int i0) {
        const int px0 = (i0 + tid) >> sh, part0 = (i0 + tid) & (pr - 1);
#pragma unroll
        for (int k = 0; k < HS; ++k)
        {
            const int i = i0 + k * NT + tid;
            if (i0 + k * NT >= pieces) continue;
            int at;
            v4i v = h[k];
            if constexpr (RG)
            {
                const int px = DivByInvariant(i, pr, t.rcp_pr), part = i - px * pr;
                if (__builtin_expect(__builtin_amdgcn_ballot_w64(back[k] != 0) != 0, 0)) v = ShiftDown16(v, back[k]);
                v ^= xm;
                if constexpr (AW) v = KeepBytes16(v, a.Ci - part * 16, a.pad_word);     // channels that do not exist count as padding in the row sum
                at = part * t.gp + px * 16;
            }
            else
            {
                v ^= xm;
                if (pow2 && pr <= NT) at = part0 * t.gp + (px0 + k * (NT >> sh)) * 16;
                else
                {
                    const int px = DivByInvariant(i, pr, t.rcp_pr);
                    at = (i - px * pr) * t.gp + px * 16;
                }
            }
            if (i < pieces) *reinterpret_cast<v4i*>(tap_lds + at) = v;
        }
    };
    load_panel(0);
    float* const tab = reinterpret_cast<float*>(tap_lds + G::Work(t.panel_bytes));
    constexpr int TP = 5 * (NCOL / 4), TS = (TP + NT - 1) / NT;
    v4i tab_piece[TS];
    const v4i pad_piece = *reinterpret_cast<const v4i*>(a.pad16);
#pragma unroll
    for (int k = 0; k < TS; ++k)
    {
        const int i = min(tid + k * NT, TP - 1), r = i / (NCOL / 4), c4 = tn * NCOL + i % (NCOL / 4) * 4;
        const float* const src = r < 4 ? a.ct.p + r * a.ct.stride : reinterpret_cast<const float*>(a.corr);
        tab_piece[k] = *reinterpret_cast<const v4i*>(src + c4);
    }
    uint32_t inside[PG];
    int lb[PG];
#pragma unroll
    for (int p = 0; p < PG; ++p)
    {
        const int from = (p & 3) * 16 + j;
        inside[p] = static_cast<uint32_t>(__shfl(static_cast<int>(taps[p >> 2]), from));
        lb[p] = (__shfl(first[p >> 2], from) - base) * 16 + (WHOLE ? g * t.gp : 0);
    }
    const int pad_at = t.gp - 16 + (WHOLE ? g * t.gp : 0);         // the last pixel of each 16 channels

    store_panel(0);
    for (int i = tid; i < pr; i += NT) *reinterpret_cast<v4i*>(tap_lds + (i + 1) * t.gp - 16) = pad_piece ^ xm;
#pragma unroll
    for (int k = 0; k < TS; ++k)
        if (tid + k * NT < TP) *reinterpret_cast<v4i*>(tab + (tid + k * NT) * 4) = tab_piece[k];
    for (int i0 = NT * HS; i0 < pieces; i0 += NT * HS)
    {
        load_panel(i0);
        store_panel(i0);
    }
    __syncthreads();

    // ---- products ---------------------------------------------------------------------------------------------------------------------
    v4i acc[CG][PG];
    int xs[PG];
#pragma unroll
    for (int p = 0; p < PG; ++p)
    {
        xs[p] = 0;
#pragma unroll
        for (int c = 0; c < CG; ++c) acc[c][p] = v4i{0, 0, 0, 0};
    }
    // where the lane reads: filter tap and, WHOLE, the k-steps left of it (the channel, else)
    int ky = t.wave_k[wk].ky, kx = t.wave_k[wk].kx, ci = t.wave_k[wk].ci + (WHOLE ? 0 : g * 16);
    int at[PG];
    auto enter_tap = [&](int skip) {
        const uint32_t bit = WHOLE || ky < a.Kh ? 1u << (ky * a.Kw + kx) : 0u;
        const int to = (ky * a.dil_y * a.W + kx * a.dil_x) * 16 + skip;
#pragma unroll
        for (int p = 0; p < PG; ++p) at[p] = (inside[p] & bit) != 0u ? lb[p] + to : pad_at + skip;
    };
    auto next_tap = [&] {
        if (++kx == a.Kw) { kx = 0; ++ky; }
    };
    int left = (tap_bytes - ci) >> 6;
    if constexpr (WHOLE) enter_tap((ci >> 4) * t.gp);
    for (int k0 = s0; k0 < s1; k0 += RD)
    {
#pragma unroll
        for (int r = 0; r < RD; ++r)
        {
            if (k0 + r >= s1) break;
            if constexpr (WHOLE)
            {
                if (left == 0)
                {
                    next_tap();
                    enter_tap(0);
                    left = tap_bytes >> 6;
                }
                --left;
            }
            else
            {
                while (ci >= tap_bytes) { ci -= tap_bytes; next_tap(); }
                enter_tap((ci >> 4) * t.gp);
                ci += 64;
            }
            v4i xb[PG];
#pragma unroll
            for (int p = 0; p < PG; ++p)
            {
                xb[p] = *reinterpret_cast<const v4i*>(tap_lds + at[p]);
                if constexpr (WHOLE) at[p] += 4 * t.gp;
            }
#pragma unroll
            for (int c = 0; c < CG; ++c)
#pragma unroll
                for (int p = 0; p < PG; ++p) acc[c][p] = __builtin_amdgcn_mfma_i32_16x16x64_i8(wv[r][c], xb[p], acc[c][p], 0, 0, 0);
            if constexpr (AW)
            {
#pragma unroll
                for (int p = 0; p < PG; ++p)
#pragma unroll
                    for (int d = 0; d < 4; ++d) xs[p] = __builtin_amdgcn_sdot4(xb[p][d], 0x01010101, xs[p], false);
            }
            if (k0 + r + RD < s1) load_weights(r);
        }
    }
    // ---- the partial tiles meet: wave (wk, wn) finishes pixel groups wk PO .. of its columns ------------------------------------------------
    constexpr int CHUNKS = NCOL / 16, NP = (PX * CHUNKS + NT - 1) / NT;
    v4i other[NP];
    const bool fuse = a.res != nullptr;
    if (fuse)
    {
#pragma unroll
        for (int i = 0; i < NP; ++i)
        {
            const int idx = tid + i * NT, r = idx / CHUNKS, chunk = idx - r * CHUNKS;
            other[i] = *reinterpret_cast<const v4i*>(a.res + static_cast<long long>(min(tm * PX + r, a.M - 1)) * a.Co + min(tn * NCOL + chunk * 16, a.Co - 16));
        }
    }
    if constexpr (AW)
    {
#pragma unroll
        for (int p = 0; p < PG; ++p)
        {
            xs[p] += __shfl_xor(xs[p], 16);
            xs[p] += __shfl_xor(xs[p], 32);
        }
    }
    __syncthreads();                                     // the panel has been read
    v4i sum[PO][CO];
    int rows[PO];
    if constexpr (WK > 1)
    {
        // [wn][finishing wave][source, without itself][PO][CO][lane]
        auto slot = [&](int to, int from) { return tap_lds + (((wm * WN + wn) * WK + to) * (WK - 1) + (from < to ? from : from - 1)) * (PO * CO * 1024) + lane * 16; };
#pragma unroll
        for (int to = 0; to < WK; ++to)
        {
            uint8_t* const d = slot(to, wk);
#pragma unroll
            for (int p = 0; p < PO; ++p)
#pragma unroll
                for (int c = 0; c < CO; ++c)
                {
                    if (to != wk) *reinterpret_cast<v4i*>(d + (p * CO + c) * 1024) = acc[G::FirstC(to) + c][G::FirstP(to) + p];
                    else sum[p][c] = acc[G::FirstC(to) + c][G::FirstP(to) + p];
                }
        }
        __syncthreads();
#pragma unroll
        for (int k = 0; k < WK - 1; ++k)
        {
            const uint8_t* const s = tap_lds + (((wm * WN + wn) * WK + wk) * (WK - 1) + k) * (PO * CO * 1024) + lane * 16;
#pragma unroll
            for (int p = 0; p < PO; ++p)
#pragma unroll
                for (int c = 0; c < CO; ++c) sum[p][c] += *reinterpret_cast<const v4i*>(s + (p * CO + c) * 1024);
        }
    }
    else
    {
#pragma unroll
        for (int p = 0; p < PO; ++p)
#pragma unroll
            for (int c = 0; c < CO; ++c) sum[p][c] = acc[c][p];
    }
    // (in the wave's own numbers, unlike FirstP and FirstC, no constants)
    const int p_first = PG >= WK ? wk * PO : wk * PG / WK, c_first = PG >= WK ? 0 : wk % (WK / PG > 0 ? WK / PG : 1) * CO;
    if constexpr (AW)
    {
        // what the bytes beyond K, and channels that do not exist, added are padding values
        const int beyond = (steps * 64 - a.Kh * a.Kw * a.Ci) * static_cast<int>(static_cast<int8_t>(a.pad_word & 0xffu));
        if constexpr (WK > 1)
        {
            __syncthreads();                             // the partial tiles have been read
            int* const rs = reinterpret_cast<int*>(tap_lds);
            if (wn == 0 && g == 0)
            {
#pragma unroll
                for (int p = 0; p < PG; ++p) rs[wk * PX + (wm * PG + p) * 16 + j] = xs[p];
            }
            __syncthreads();
#pragma unroll
            for (int p = 0; p < PO; ++p)
            {
                rows[p] = -beyond;
#pragma unroll
                for (int k = 0; k < WK; ++k) rows[p] += rs[k * PX + (wm * PG + p_first + p) * 16 + j];
            }
        }
        else
        {
#pragma unroll
            for (int p = 0; p < PO; ++p) rows[p] = xs[p] - beyond;
        }
    }
    if constexpr (WK > 1) __syncthreads();               // all partial sums have been read; the outputs take their place
    WithBits(a.rq, [&](auto bits) {
        constexpr bool kBits = decltype(bits)::value;
        const int cl = (wn * CG + c_first) * 16 + 4 * g;
        uint8_t* const out_at = tap_lds + ((wm * PG + p_first) * 16 + j) * OP + cl;
        if constexpr (PO >= CO)
        {
#pragma unroll
            for (int c = 0; c < CO; ++c)
            {
                const v4i corr = *reinterpret_cast<const v4i*>(tab + 4 * NCOL + cl + 16 * c);
                const Fast4 f = {*reinterpret_cast<const float4*>(tab + 2 * NCOL + cl + 16 * c), *reinterpret_cast<const float4*>(tab + 3 * NCOL + cl + 16 * c)};
                v4i v[PO];
                uint32_t out[PO];
#pragma unroll
                for (int p = 0; p < PO; ++p) v[p] = sum[p][c] + corr + (AW ? rows[p] * a.zw_neg : 0);
                RequantPixels<kBits, PO>(v, out, f, ChanTab{tab, NCOL}, cl + 16 * c, a.rq);
#pragma unroll
                for (int p = 0; p < PO; ++p) *reinterpret_cast<uint32_t*>(out_at + p * 16 * OP + 16 * c) = out[p];
            }
        }
        else
        {
            Fast4 f[CO];
            v4i corr[CO];
#pragma unroll
            for (int c = 0; c < CO; ++c)
            {
                corr[c] = *reinterpret_cast<const v4i*>(tab + 4 * NCOL + cl + 16 * c);
                f[c] = {*reinterpret_cast<const float4*>(tab + 2 * NCOL + cl + 16 * c), *reinterpret_cast<const float4*>(tab + 3 * NCOL + cl + 16 * c)};
            }
#pragma unroll
            for (int p = 0; p < PO; ++p)
            {
                v4i v[CO];
                uint32_t out[CO];
#pragma unroll
                for (int c = 0; c < CO; ++c) v[c] = sum[p][c] + corr[c] + (AW ? rows[p] * a.zw_neg : 0);
                RequantChannels<kBits, CO, 16>(v, out, f, ChanTab{tab, NCOL}, cl, a.rq);
#pragma unroll
                for (int c = 0; c < CO; ++c) *reinterpret_cast<uint32_t*>(out_at + p * 16 * OP + 16 * c) = out[c];
            }
        }
    });
    __syncthreads();
    const OutPtr outp = MakeOutPtr(a.y, static_cast<long long>(a.M) * a.Co);
#pragma unroll
    for (int i = 0; i < NP; ++i)
    {
        const int idx = tid + i * NT, r = idx / CHUNKS, chunk = idx - r * CHUNKS;
        const int m = tm * PX + r, c0 = tn * NCOL + chunk * 16;
        if ((PX * CHUNKS % NT == 0 || r < PX) && m < a.M && c0 < a.Co)
        {
            v4i v = *reinterpret_cast<const v4i*>(tap_lds + r * OP + chunk * 16);
            if (fuse) v = AddQuantize16Dev(v, other[i], a.add);
            if (a.vec_out) StoreOut16(outp, static_cast<long long>(m) * a.Co + c0, v);
            else StoreRagged16(a.y + static_cast<long long>(m) * a.Co + c0, v, a.Co - c0);
        }
    }
}

// KG, BM, BN: one of TapTile's.
template <int KG, int BM, int BN, bool AW, bool RG, bool WHOLE>
__global__ __launch_bounds__((64 * TapTile<KG, BM, BN>::WAVES), (TapTile<KG, BM, BN>::WAVES_PER_SIMD)) void TapPanelKernel(TapPanelArgs t)
{
    using T = TapTile<KG, BM, BN>;
    TapPanelBlock<T::WM, T::WN, KG, T::CG, T::PG, T::RD, AW, RG, WHOLE>(t);
}

} // namespace mi355x
