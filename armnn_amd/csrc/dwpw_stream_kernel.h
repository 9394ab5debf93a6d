// Depthwise 3x3 (stride 1 or 2) + the pointwise 1x1 convolution that consumes it as ONE kernel, for the wide, shallow
// layers at the front of a MobileNet: 32, 64 or 128 channels between the layers, 64, 128 or 256 output channels.
//
// Run apart, these layers are bound by memory: the tensor between them is written once and read once (112 x 112 x 32 at 64
// images: 26 MB each way, next to 26 MB in and 51 MB out).  Here it never leaves the CU.
//   * A block of four (or eight) waves is persistent: its waves keep the pointwise weights and both layers' constants in registers for
//     their whole life and walk items -- TH x TW output pixels of one image over ALL channels -- with the next item's input
//     halo in flight (in registers) while the current one is computed.  Two barriers per item: halo staged / panel complete.
//   * Depthwise phase: the matrix-core arithmetic of DepthwiseMfmaKernel (16 channels x 16 pixels x 4 taps per
//     v_mfma_i32_16x16x64_i8 over diagonal weight operands kept in registers), requantized with the depthwise layer's own
//     constants; the codes -- the bytes the separate layer would have stored, shifted to int8 where they are uint8 -- go
//     to an LDS panel [pixel][channel].
//   * Pointwise phase: a wave owns 64 output channels of its share of the pixels, as 16 x 16 results with pixels as rows; column j of the
//     four results of 16 pixels is channel 4 j + result, so that a lane holds channels 4 j .. 4 j + 3 of four pixels, always the
//     same four channels: weights (8 to 32 registers) and constants stay where they are.  (With channels as rows, 32 x 32, a wave
//     read weights and constants again for every item, a third of the LDS traffic; a pass of
//     MobileNetV1 at 64 images 160.7 -> 158.0 us, at 256 576 -> 569.5.)  The requantized dwords pass
//     through a wave-private LDS area and leave as 16 bytes per lane.
//   * Loads and stores of a wave complete in issue order and share one counter: an item's stores are issued at the start of
//     the next iteration, ahead of that iteration's loads, so the wait for those loads covers nothing younger.
//   * Stores go through a buffer descriptor of the item's image: a pixel right of the image gets an offset past the
//     descriptor's size, a row below the image runs past it by itself, and the hardware drops those stores.
// Both layers' arithmetic is untouched -- exact int32 sums, the same requantization routine with the same constants -- so
// the bytes are those of the two layers run one after the other.
#pragma once

#include <hip/hip_runtime.h>

#include "common.h"
#include "conv_kernels.h"
#include "device_math.h"
#include "dw_mfma_kernel.h"

namespace mi355x
{

struct DwPwStreamArgs
{
    // depthwise 3x3, multiplier 1
    const uint8_t*  x;
    const uint8_t*  pad16;      // 16 bytes that become the depthwise padding value under dw_xor
    const uint32_t* wpack;      // [C][4] dwords, rows of the 3x3 filter per channel (Dw3x3Args::wpack)
    ChanTab         dw_ct;
    const int32_t*  dw_corr;
    int N, H, W, Ho, Wo;
    int pad_top, pad_left;
    int tiles_x, tiles_y;
    int total_items, xcd_chunk;
    uint32_t rcp_tiles_x, rcp_tiles_y;
    uint32_t dw_xor;
    Requant dw_rq;
    // pointwise 1x1
    const int8_t*  w;           // [Co_pad][w_stride]
    int            w_stride;
    ChanTab        pw_ct;
    const int32_t* pw_corr;
    uint8_t*       y;
    uint32_t       mid_xor;     // 0x80808080 when the tensor between the layers is uint8: the panel holds the int8-shifted codes
    Requant        pw_rq;
};

// S: depthwise stride; C: channels between the layers; NO: output channels; TH x TW: output pixels per item; NWAVES: 4 or
// 8 waves per block (8 for 256 output channels: two to each 64 of them)
template <int S, int C, int NO, int TH, int TW, int NWAVES = 4>
struct DwPwStreamGeom
{
    static_assert(C == 32 || C == 64 || C == 128 || C == 256, "channels between the layers");
    static_assert(NO == 64 || NO == 128 || NO == 256, "output channels");
    static_assert(TW == 8 || TW == 16, "a group of 16 pixels is one or two whole tile rows");
    static constexpr int NW = NWAVES, NT = 64 * NW;
    static constexpr int NCG = C / 16;
    static constexpr int P = TH * TW;                     // pixels per item
    static_assert(P % 64 == 0, "groups of 16 pixels, shared evenly by four waves");
    static constexpr int NPG = P / 16;
    static constexpr int CGW = NCG > NW ? NCG / NW : 1;  // channel groups per wave
    static constexpr int WPC = NCG < NW ? NW / NCG : 1;  // waves sharing a channel group (they split the pixel groups)
    static constexpr int UNITS = NPG / WPC;               // pixel groups per wave and channel group
    static_assert(NPG % WPC == 0, "pixel groups split evenly");
    static constexpr int HR = (TH - 1) * S + 3;
    static constexpr int HC = (TW - 1) * S + 3;
    static constexpr int PITCH = C + 16;
    static constexpr int ROWP_RAW = HC * PITCH;
    static constexpr int ROWP = (TW == 8 && S == 1) ? ((ROWP_RAW + 127) / 256 * 256 + 128) : ROWP_RAW;
    static constexpr int HALO = HR * ROWP;                // the halo buffer
    static constexpr int KP = C + 16;                     // bytes per panel row
    static constexpr int PANEL = P * KP;
    static constexpr int TAB = 2 * NO * 4 + 2 * C * 4;    // mult and biasf of both layers
    static constexpr int WN = NO / 64, WM = NW / WN;      // waves side by side over channels and pixels
    static_assert(NW % WN == 0 && P % (16 * WM) == 0, "whole shares");
    static constexpr int PXW = P / WM, MT = PXW / 16;     // a wave's pixels, in groups of 16
    static constexpr int KB = C >= 64 ? 64 : 32, KST = C / KB;     // bytes of K per MFMA
    static constexpr int LDO = 64 + 16;
    static constexpr int OUT = NW * PXW * LDO;
    static constexpr int QUADS = PXW * 4 / 64;            // 16-byte stores per lane and item
    static constexpr int SMEM = HALO + PANEL + TAB + OUT;
    // Blocks per CU that LDS allows; the register budget follows it (a few spilled registers cost less than the third block
    // gains: 112 x 112 x 32 -> 64 at 64 images 29.5 us with two blocks, 24.4 with three).
    // (With 128 channels the weights and constants alone take 60 registers: a third block of four waves would spill 88, a second of
    // eight took a launch of one image from 6.2 to 12.1 us.)
    static constexpr int FIT = 160 * 1024 / SMEM, MOST = C <= 64 ? 3 : NWAVES == 4 ? 2 : 1;
    static constexpr int BLOCKS = FIT >= MOST ? MOST : FIT >= 1 ? FIT : 1;
    static constexpr int WAVES_PER_SIMD = BLOCKS * NW / 4;
};

template <int S, int C, int NO, int TH, int TW, int NWAVES = 4>
__global__ __launch_bounds__(64 * NWAVES)
__attribute__((amdgpu_waves_per_eu(DwPwStreamGeom<S, C, NO, TH, TW, NWAVES>::WAVES_PER_SIMD, DwPwStreamGeom<S, C, NO, TH, TW, NWAVES>::WAVES_PER_SIMD)))
void DwPwStreamKernel(DwPwStreamArgs a)
{
    using G = DwPwStreamGeom<S, C, NO, TH, TW, NWAVES>;
    constexpr int NW = G::NW;
    constexpr int NT = G::NT, NCG = G::NCG, HR = G::HR, HC = G::HC, PITCH = G::PITCH, ROWP = G::ROWP, HALO = G::HALO;
    constexpr int CGW = G::CGW, WPC = G::WPC, UNITS = G::UNITS, KP = G::KP, LDO = G::LDO, QUADS = G::QUADS;
    constexpr int RPG = 16 / TW;
    // pixel groups whose depthwise outputs are computed together (a pass at 64 images: 4 170.8, 2 171.3, 1 172.1 us)
    constexpr int UB = UNITS % 4 == 0 ? 4 : UNITS % 2 == 0 ? 2 : 1;
    constexpr int CPP = C / 16;
    constexpr int NCH = HR * HC * CPP;
    constexpr int NST = (NCH + NT - 1) / NT;
    extern __shared__ __attribute__((aligned(16))) uint8_t dwpw_stream_lds[];
    uint8_t* const lds = dwpw_stream_lds;
    constexpr int PANEL0 = HALO, TAB0 = PANEL0 + G::PANEL, OUT0 = TAB0 + G::TAB;

    const int tid = threadIdx.x;
    const int lane = tid & 63, wave = tid >> 6;
    const int xcd = blockIdx.x & 7;
    const int step = static_cast<int>(gridDim.x >> 3);
    const int item_end = min((xcd + 1) * a.xcd_chunk, a.total_items);
    int item = xcd * a.xcd_chunk + static_cast<int>(blockIdx.x >> 3);
    if (item >= item_end) return;

    // ---- what the exact path reads of both layers' tables ------------------------------------------------------------------
    for (int i = tid; i < NO / 2; i += NT)
        *reinterpret_cast<v4i*>(lds + TAB0 + i * 16) = *reinterpret_cast<const v4i*>(a.pw_ct.p + i / (NO / 4) * a.pw_ct.stride + i % (NO / 4) * 4);
    for (int i = tid; i < C / 2; i += NT)
        *reinterpret_cast<v4i*>(lds + TAB0 + 2 * NO * 4 + i * 16) = *reinterpret_cast<const v4i*>(a.dw_ct.p + i / (C / 4) * a.dw_ct.stride + i % (C / 4) * 4);
    const ChanTab pw_exact{reinterpret_cast<const float*>(lds + TAB0), NO}, dw_exact{reinterpret_cast<const float*>(lds + TAB0) + 2 * NO, C};

    // ---- staging of the input halo (as in DepthwiseMfmaKernel, all C channels) -------------------------------------------
    const int dxm = static_cast<int>(a.dw_xor);
    const int in_image = a.H * a.W * C;
    int st_lds[NST], st_row[NST], st_col[NST], st_off[NST];
#pragma unroll
    for (int k = 0; k < NST; ++k)
    {
        const int i = min(tid + k * NT, NCH - 1);
        const int part = i % CPP;
        const int pix = i / CPP;
        st_col[k] = pix % HC;
        st_row[k] = pix / HC;
        st_lds[k] = st_row[k] * ROWP + st_col[k] * PITCH + part * 16;
        st_off[k] = (st_row[k] * a.W + st_col[k]) * C + part * 16;
        if (tid + k * NT >= NCH) st_lds[k] = -1;
    }
    v4i st[NST];
    struct Where { int tx, ty, n; };
    auto decode = [&](int b) {
        Where w;
        int q = DivByInvariant(b, a.tiles_x, a.rcp_tiles_x);
        w.tx = b - q * a.tiles_x; b = q;
        q = DivByInvariant(b, a.tiles_y, a.rcp_tiles_y);
        w.ty = b - q * a.tiles_y; w.n = q;
        return w;
    };
    auto issue = [&](int b) {
        const Where w = decode(b);
        const int iy_org = w.ty * TH * S - a.pad_top;
        const int ix_org = w.tx * TW * S - a.pad_left;
        const uint8_t* xn = a.x + static_cast<long long>(w.n) * in_image;
        const int org = (iy_org * a.W + ix_org) * C;
#pragma unroll
        for (int k = 0; k < NST; ++k)
        {
            const bool ok = static_cast<unsigned>(iy_org + st_row[k]) < static_cast<unsigned>(a.H) &&
                            static_cast<unsigned>(ix_org + st_col[k]) < static_cast<unsigned>(a.W);
            const uint8_t* src = ok ? xn + (org + st_off[k]) : a.pad16;
            st[k] = *reinterpret_cast<const v4i*>(src);
        }
    };
    auto commit = [&](int halo) {
#pragma unroll
        for (int k = 0; k < NST; ++k)
            if (st_lds[k] >= 0) *reinterpret_cast<v4i*>(lds + halo + st_lds[k]) = st[k] ^ dxm;
    };

    // The first item's halo is requested ahead of the constants: it is wanted first, and loads arrive in the order of their requests.
    issue(item);

    // ---- depthwise roles: lane (j, g): pixel j of a group of 16 and tap slot g as an operand, channel quad g as a result --
    const int j = lane & 15, g = lane >> 4;
    const int rj = j / TW, cj = j % TW;
    const int cg0 = NCG > NW ? wave * CGW : wave % NCG;
    const int pg0 = NCG > NW ? 0 : wave / NCG;
    int lds_tap[3];
    v4i wa[CGW][3], corr4[CGW];
    Fast4 f4[CGW];
    {
        int wrow[3], wshift[3];
#pragma unroll
        for (int m = 0; m < 3; ++m)
        {
            const int t = 4 * m + g;
            const int tc = min(t, 8);                      // slots past the ninth tap read the ninth; their weights are zero
            lds_tap[m] = ((pg0 * RPG + rj) * S + tc / 3) * ROWP + (cj * S + tc % 3) * PITCH + cg0 * 16;
            wrow[m] = tc / 3;
            wshift[m] = t < 9 ? 8 * (tc % 3) : 24;         // shift 24: the zero byte of a packed filter row
        }
#pragma unroll
        for (int i = 0; i < CGW; ++i)
        {
            const int c0 = (cg0 + i) * 16;
            const uint4 w4 = *reinterpret_cast<const uint4*>(a.wpack + (c0 + j) * 4);
            const int dw = j >> 2, sh = 8 * (j & 3);
#pragma unroll
            for (int m = 0; m < 3; ++m)
            {
                const uint32_t ra = wrow[m] == 0 ? w4.x : wrow[m] == 1 ? w4.y : w4.z;
                const int ba = static_cast<int>(((ra >> wshift[m]) & 0xffu) << sh);
                wa[i][m] = v4i{dw == 0 ? ba : 0, dw == 1 ? ba : 0, dw == 2 ? ba : 0, dw == 3 ? ba : 0};
            }
            corr4[i] = *reinterpret_cast<const v4i*>(a.dw_corr + c0 + 4 * g);
            f4[i] = LoadFast4(a.dw_ct, c0 + 4 * g);
        }
    }
    // the codes of pixel (pg0 + u WPC) 16 + j, channels (cg0 + i) 16 + 4 g ..: one dword of the panel
    const int panel_write = PANEL0 + (pg0 * 16 + j) * KP + cg0 * 16 + 4 * g;

    // ---- pointwise roles: the wave's pixels [px0, px0 + PXW) and channels [n0, n0 + 64); lane (j, g): operand row or column j, bytes of K
    // by g; as a result channels n0 + 4 j .. + 3 of pixels 4 g .. 4 g + 3 of a group of 16 ----------------------------------
    constexpr int WN = G::WN, PXW = G::PXW, MT = G::MT, KB = G::KB, KST = G::KST, KL = KB / 4;    // KL: a lane's bytes of K
    const int px0 = wave / WN * PXW, n0 = wave % WN * 64;
    typedef typename std::conditional<KB == 64, v4i, long>::type KVec;
    KVec pw[KST][4];
    v4i pw_init[4];
    Fast4 pf;
#pragma unroll
    for (int t = 0; t < 4; ++t)
    {
#pragma unroll
        for (int ks = 0; ks < KST; ++ks)
            pw[ks][t] = *reinterpret_cast<const KVec*>(a.w + static_cast<long long>(n0 + 4 * j + t) * a.w_stride + ks * KB + g * KL);
        const int c = a.pw_corr[n0 + 4 * j + t];
        pw_init[t] = v4i{c, c, c, c};
    }
    pf = LoadFast4(a.pw_ct, n0 + 4 * j);
    const int a_frag = PANEL0 + (px0 + j) * KP + g * KL;
    // the wave's output area [PXW pixels][LDO]
    const int out_area = OUT0 + wave * PXW * LDO;
    const int out_write = out_area + 4 * g * LDO + 4 * j;
    // 16-byte pieces of that area: piece id = k 64 + lane -> (pixel id / 4, part id % 4).  16 pixels per store instruction are whole
    // tile rows, so a lane keeps its column and part; only the row moves with k.
    constexpr int RPS = 16 / TW;                           // tile rows per store instruction
    const int sr0 = lane / 4, part0 = lane % 4;
    const int y_col = sr0 % TW;
    const int out_read = out_area + sr0 * LDO + part0 * 16;
    const int y_lane = (((px0 + sr0) / TW) * a.Wo + y_col) * NO + n0 + part0 * 16;
    const int y_step = RPS * a.Wo * NO;
    const int image_bytes = a.Ho * a.Wo * NO;

    int out_base = 0, out_n = -1, out_cols = 0;
    auto store_outputs = [&]() {
        const __amdgpu_buffer_rsrc_t yrsrc = __builtin_amdgcn_make_buffer_rsrc(a.y + static_cast<long long>(out_n) * image_bytes, 0, image_bytes, 0x00020000);
#pragma unroll
        for (int k = 0; k < QUADS; ++k)
        {
            const v4i v = *reinterpret_cast<const v4i*>(lds + out_read + k * 16 * LDO);
            const int yo = y_col < out_cols ? out_base + y_lane + k * y_step : static_cast<int>(0x80000000u);
            __builtin_amdgcn_raw_buffer_store_b128(v, yrsrc, yo, 0, 0);
        }
    };
    auto depthwise = [&](int halo) {
#pragma unroll
        for (int i = 0; i < CGW; ++i)
#pragma unroll
            for (int u0 = 0; u0 < UNITS; u0 += UB)
            {
                v4i acc[UB];
                uint32_t q[UB];
#pragma unroll
                for (int k = 0; k < UB; ++k)
                {
                    const int lo = halo + i * 16 + (u0 + k) * (WPC * RPG * S * ROWP);
                    const v4i b0 = *reinterpret_cast<const v4i*>(lds + lds_tap[0] + lo);
                    const v4i b1 = *reinterpret_cast<const v4i*>(lds + lds_tap[1] + lo);
                    const v4i b2 = *reinterpret_cast<const v4i*>(lds + lds_tap[2] + lo);
                    acc[k] = corr4[i];
                    acc[k] = __builtin_amdgcn_mfma_i32_16x16x64_i8(wa[i][0], b0, acc[k], 0, 0, 0);
                    acc[k] = __builtin_amdgcn_mfma_i32_16x16x64_i8(wa[i][1], b1, acc[k], 0, 0, 0);
                    acc[k] = __builtin_amdgcn_mfma_i32_16x16x64_i8(wa[i][2], b2, acc[k], 0, 0, 0);
                }
                RequantPixels<true, UB>(acc, q, f4[i], dw_exact, (cg0 + i) * 16 + 4 * g, a.dw_rq);
#pragma unroll
                for (int k = 0; k < UB; ++k) *reinterpret_cast<uint32_t*>(lds + panel_write + i * 16 + (u0 + k) * (WPC * 16 * KP)) = q[k] ^ a.mid_xor;
            }
    };
    auto pointwise = [&](int b) {
        const Where w = decode(b);
        out_base = ((w.ty * TH) * a.Wo + w.tx * TW) * NO;
        out_cols = a.Wo - w.tx * TW;
        out_n = w.n;
        WithBits(a.pw_rq, [&](auto bits) {
#pragma unroll
            for (int mt = 0; mt < MT; ++mt)
            {
                v4i acc[4];
#pragma unroll
                for (int ks = 0; ks < KST; ++ks)
                {
                    const KVec x = *reinterpret_cast<const KVec*>(lds + a_frag + mt * 16 * KP + ks * KB);
#pragma unroll
                    for (int t = 0; t < 4; ++t)
                    {
                        if constexpr (KB == 64) acc[t] = __builtin_amdgcn_mfma_i32_16x16x64_i8(x, pw[ks][t], ks == 0 ? pw_init[t] : acc[t], 0, 0, 0);
                        else acc[t] = __builtin_amdgcn_mfma_i32_16x16x32_i8(x, pw[ks][t], ks == 0 ? pw_init[t] : acc[t], 0, 0, 0);
                    }
                }
                v4i v[4];
                uint32_t out[4];
#pragma unroll
                for (int r = 0; r < 4; ++r) v[r] = v4i{acc[0][r], acc[1][r], acc[2][r], acc[3][r]};
                RequantPixels<decltype(bits)::value, 4>(v, out, pf, pw_exact, n0 + 4 * j, a.pw_rq);
#pragma unroll
                for (int r = 0; r < 4; ++r) *reinterpret_cast<uint32_t*>(lds + out_write + (mt * 16 + r) * LDO) = out[r];
            }
        });
    };

    while (true)
    {
        // (one halo buffer: its readers, the depthwise phase of the item before, all passed that item's second barrier)
        commit(0);
        // all waves are done with the item before (its panel has been multiplied) and this item's halo is in LDS; on the first
        // pass the barrier also orders the resident weights and table rows before their first use
        __syncthreads();
        // the item before leaves its wave-private area (LDS operations of a wave complete in order: no barrier needed), ahead
        // of the next loads
        if (out_n >= 0) store_outputs();
        const int next = item + step;
        const bool more = next < item_end;
        if (more) issue(next);
        depthwise(0);
        __syncthreads();                                   // the panel is complete
        pointwise(item);
        if (!more) break;
        item = next;
    }
    store_outputs();
}

} // namespace mi355x
