#include "tap_panel.h"

#include <algorithm>

#include "common.h"
#include "igemm.h"
#include "igemm_tile.h"
#include "tap_panel_kernel.h"
#include "tap_panel_run.h"

using namespace mi355x;

namespace
{
constexpr int kLdsBytes = 160 * 1024, kTapTiles = 8;

TapWindow Window(const ConvGeom& g) { return {g.H, g.W, g.Ho, g.Wo, g.Kh, g.Kw, g.stride_y, g.stride_x, g.dil_y, g.dil_x}; }

// Bytes per 16 channels of the panel of `pixels` outputs, one pixel of padding with them, made an odd number of pixels.
int PanelPitch(const ConvGeom& g, long long M, int pixels)
{
    const long long run = TapRun(Window(g), M, pixels);
    return run > kLdsBytes / 16 ? kLdsBytes : static_cast<int>((run + 1) | 1) * 16;
}

// What a launch on a tile takes, in clocks: from its start to its end, and of all 256 CUs together, per CU.  Negative: the tile does not fit.
// alone_in_turns: a CU holds one block at a time and gets several.
// us: microseconds of the launch by itself.  bringing: the panel's share of its blocks' work.
struct Account { double span, work, us, bringing; bool alone_in_turns; };

// A block takes 4900 clocks of round trips and set-up, 6.6 for the pieces a lane brings to the panel, and for each k-step a wave takes 16 per matrix
// instruction and 130 beside them; partial tiles cost 43 per four results and further wave of K.  Blocks of a CU overlap until its SIMDs are full of
// matrix instructions, write-out (90), partial tiles and the panel.  Fitted to 60 layers of 3x3 and 5x5 taps, strides 1 and 2, 16 to 512
// channels and over 392 tiles of 32 x 32, each on six to eight tiles: spans are 14 % off, but the tile with the least one takes 1.3 % longer than the best.
// The microseconds are a sum of the same parts fitted to 508 layers with filters of 2 to 32 taps and dilations 1 to 6 as well: 10 % off.
template <int KG, int BM, int BN>
Account TileAccount(const mi355x_conv2d_s* p, long long M, int steps)
{
    using T = TapTile<KG, BM, BN>;
    using G = typename T::Geom;
    constexpr Account none = {-1.0, -1.0, 0.0, 0.0, false};
    const ConvGeom& g = p->geom;
    if (p->Co_pad % BN != 0) return none;
    const double panel = static_cast<double>((p->ragged_ck ? p->ragged_ck : g.Ci) / 16) * PanelPitch(g, M, BM);
    if (panel > kLdsBytes) return none;
    const int smem = G::Smem(static_cast<int>(panel));
    const int resident = smem > kLdsBytes ? 0 : std::min(kLdsBytes / smem, T::WAVES_PER_SIMD * 4 / T::WAVES);
    if (resident == 0) return none;
    constexpr double kPerSimd = T::WAVES / 4.0, kMfma = 16.0 * T::CG * T::PG, kPartial = 43.0 * (KG - 1) * T::CG * T::PG / 4.0;
    const double k = (steps + KG - 1) / KG, bring = panel / 256 * 6.6;
    const double block = 4900.0 + bring / kPerSimd + k * (kMfma + 130.0) + kPartial;
    const double share = kPerSimd * (k * kMfma + 90.0 + kPartial) + bring;
    const auto round = [&](long long blocks) { return blocks == 0 ? 0.0 : std::max(block, blocks * share + 4900.0); };
    const long long blocks = (M + BM - 1) / BM * ((g.Co + BN - 1) / BN), slots = 256ll * resident;
    const double rounds = static_cast<double>((blocks + slots - 1) / slots), per_cu = blocks / 256.0, mfma = k * T::CG * T::PG;
    const double us = 2.53 + rounds * (1.37 + 0.0156 * mfma + 0.0518 * k + 3.02e-5 * panel / kPerSimd) + per_cu * (kPerSimd * (0.0112 * mfma + 0.13) + 4.65e-6 * panel);
    return {static_cast<double>(blocks / slots) * round(resident) + round((blocks % slots + 255) / 256), blocks * share / 256.0, us, bring / share, resident == 1 && blocks > 256};
}

// Whether 256-row tiles of one wave per SIMD, `columns` channels wide, fill the chip (RunPlan gives them such launches).
bool Fill256Rows(const mi355x_conv2d_s* p, long long M, int columns) { return p->Co_pad % columns == 0 && (M + 255) / 256 * (p->Co_pad / columns) >= 224; }

// Microseconds that a launch of over kSmallConvMostTiles tiles takes on the kernels which walk k-tiles and read pixels per tap, wherever the taps are: a line for each
// tile, fitted to 530 layers of 3 to 32 taps, 16 to 1024 channels and dilations 1 to 6, 10 % off.
double TiledUs(const mi355x_conv2d_s* p, long long M)
{
    struct Line { int bm, bn, bk; double launch, k_tile, k_tile_of_round, round; };      // a round: 256 blocks
    const ConvGeom& g = p->geom;
    const int K = g.Kh * g.Kw * (p->ragged_ck ? p->ragged_ck : g.Ci);
    const auto us = [&](const Line& l) {
        const double rounds = static_cast<double>((M + l.bm - 1) / l.bm * ((g.Co + l.bn - 1) / l.bn)) / 256.0, k_tiles = (K + l.bk - 1) / l.bk;
        return l.launch + k_tiles * (l.k_tile + rounds * l.k_tile_of_round) + rounds * l.round;
    };
    if (g.Ci % 128 == 0)
    {
        if (Fill256Rows(p, M, 256) || Fill256Rows(p, M, 128)) return us({256, 128, 128, 9.06, 0.0, 0.729, 12.4});
        const bool one_round = (M + 63) / 64 * ((g.Co + 63) / 64) <= 256;                // three stages of k-tiles
        return us({64, 64, 128, one_round ? 3.01 : 1.71, 0.29, 0.145, 1.11});
    }
    if (IgemmTile(0, false, M, g.Co, p->Co_pad) == 64) return us({64, 64, 64, 2.37, 0.308, 0.0647, 0.57});
    return g.Co <= 64 ? us({128, 64, 64, 2.45, 0.23, 0.183, 0.82}) : us({128, 128, 64, 3.71, 0.09, 0.31, 1.48});
}

template <int KG, int BM, int BN, bool AW, bool RG, bool WHOLE>
int LaunchT(const mi355x_conv2d_s* p, uint32_t batch, const void* x, void* y, const uint8_t* res, const AddFuse* add, hipStream_t stream)
{
    using T = TapTile<KG, BM, BN>;
    using G = typename T::Geom;
    const ConvGeom& g = p->geom;
    TapPanelArgs t;
    bool unit_fast = false;
    if (const int rc = FillIgemmLdsArgs(p, G::PX, G::NCOL, batch, x, y, &t.g, &unit_fast)) return rc;
    IgemmArgs& a = t.g;
    a.w = p->w_frag;
    a.vec_out = (g.Co & 15) == 0 && (reinterpret_cast<uintptr_t>(y) & 15) == 0;
    if (res) { a.res = res; a.add = *add; }
    const long long in_pixels = static_cast<long long>(batch) * g.H * g.W;
    if (RG)
    {
        a.Ck = p->ragged_ck;
        a.x_last16 = a.x + in_pixels * g.Ci - 16;
    }
    const long long nblocks = static_cast<long long>(a.tiles_m) * a.tiles_n;
    const int tap_bytes = RG ? a.Ck : a.Ci, pr = tap_bytes / 16;
    t.gp = PanelPitch(g, a.M, G::PX);
    t.panel_bytes = pr * t.gp;
    const int smem = G::Smem(t.panel_bytes);
    t.in_pixels = static_cast<int>(in_pixels);
    const auto reciprocal = [](int d) { return static_cast<uint32_t>((0x100000000ull + static_cast<uint32_t>(d) - 1) / static_cast<uint32_t>(d)); };
    t.tap_rows = 0;
    for (int ky = 0; ky < g.Kh; ++ky) t.tap_rows |= 1u << (ky * g.Kw);
    t.rcp_pr = reciprocal(pr);
    t.by_columns = static_cast<long long>(p->Co_pad) * p->K_pad > 2 * in_pixels * g.Ci && nblocks * a.tiles_m < (1ll << 32);
    t.minor = t.by_columns ? a.tiles_m : a.tiles_n;
    t.rcp_minor = reciprocal(t.minor);
    if (g.Kh == 1) a.dil_y = 1;                          // (one row has none, whatever the descriptor says: the kernel counts its reach in taps)
    if (g.Kw == 1) a.dil_x = 1;
    t.rcp_dy = reciprocal(a.dil_y);
    t.rcp_dx = reciprocal(a.dil_x);
    a.wo_magic = reciprocal(a.Wo);
    a.ho_magic = reciprocal(a.Ho);
    const int steps = (a.Kh * a.Kw * tap_bytes + 63) / 64;
    for (int w = 0; w <= KG; ++w)
    {
        const int step = steps * w / KG, tap = step * 64 / tap_bytes;
        t.wave_k[w] = {step, tap / a.Kw, tap % a.Kw, step * 64 % tap_bytes};
    }
    const auto kernel = TapPanelKernel<KG, BM, BN, AW, RG, WHOLE>;
    static const hipError_t attr = hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, kLdsBytes);
    MI355X_HIP(attr);
    NoteKernel("TapPanelKernel<%d, %d, %d, %s, %s, %s>", KG, BM, BN, BoolName(AW), BoolName(RG), BoolName(WHOLE));
    hipLaunchKernelGGL(kernel, dim3(static_cast<unsigned>((nblocks + 7) / 8 * 8)), dim3(64 * T::WAVES), smem, stream, t);
    MI355X_HIP(hipGetLastError());
    return 0;
}

bool Unit(const ConvGeom& g)
{
    return g.Kh == 1 && g.Kw == 1 && g.stride_x == 1 && g.stride_y == 1 && g.pad_top == 0 && g.pad_left == 0 && g.Ho == g.H && g.Wo == g.W;
}

int KSteps(const mi355x_conv2d_s* p) { return (p->geom.Kh * p->geom.Kw * (p->ragged_ck ? p->ragged_ck : p->geom.Ci) + 63) / 64; }
} // namespace

bool mi355x::TapPanelTakes(const mi355x_conv2d_s* p)
{
    const ConvGeom& g = p->geom;
    if (Unit(g)) return static_cast<long long>((p->ragged_ck ? p->ragged_ck : g.Ci) / 16) * PanelPitch(g, 32, 32) <= kLdsBytes - 4096;
    // (a bit per tap; below seven k-steps the kernels with few instructions ahead of their loads are as fast: 3 x 3 over 16 channels 0.85 to 0.98 of
    // their rate here, over 32 0.82 to 1.05, over 48 1.04 to 1.27)
    return g.Kh * g.Kw > 1 && g.Kh * g.Kw <= 32 && TapsInOrder(Window(g)) && KSteps(p) >= 7 &&
           static_cast<long long>((p->ragged_ck ? p->ragged_ck : g.Ci) / 16) * PanelPitch(g, 32, 32) <= kLdsBytes - 4096;
}

int mi355x::TapPanelTile(const mi355x_conv2d_s* p, uint32_t batch)
{
    const ConvGeom& g = p->geom;
    if (!p->w_frag || !TapPanelTakes(p)) return -1;
    const long long M = static_cast<long long>(batch) * g.Ho * g.Wo, in_pixels = static_cast<long long>(batch) * g.H * g.W, columns = (g.Co + 31) / 32;
    const long long tiles = (M + 31) / 32 * columns;
    // (pixels and tiles are decoded with reciprocals)
    if (in_pixels > (1ll << 30) || M > (1ll << 30) || M * std::max(g.Wo, g.Ho) >= (1ll << 32) || tiles * columns >= (1ll << 32) || (Unit(g) && M >= 65536)) return -1;
    const int steps = KSteps(p);
    if (Unit(g) && p->tile_override == 0)
    {
        // 1x1 layers, two stretches between other kernels.  Over 256 tiles of 32 x 32, which SmallConvKernel runs in a second round of one per CU, 32 x 64
        // tiles of eight waves are half as many (300 rows 768 -> 1024 4.57 -> 4.21 us, 1024 -> 1024 5.54 -> 4.48, 2048 -> 1024 7.78 -> 5.69; 400 rows 2048 ->
        // 1001 8.36 -> 6.43; 512 rows 2048 -> 1024 8.36 -> 7.38, but 1024 -> 1024 5.26 against 5.40, 64 rows 2048 -> 4096, 256 tiles, 6.04 against 6.45).
        // From 28 k-steps on that is so for all layers (of 320 drawn ones 0.66 to 1.04 of the time), and over kSmallConvMostTiles, where the other side is a larger tile
        // (1107 rows 736 -> 384 6.13 -> 4.84).  Below, of those whose steps lie whole in the channels, if few of the 64 columns are idle (0.74 to 1.07; 2977 rows
        // 1344 -> 96 4.96 against 5.29, 1690 rows 1088 -> 144 4.90 against 5.38); the others, whose steps find their place anew each, at few rows, whose
        // weights outweigh them by far, from 16 k-steps or a good part of a second round on (85 rows 1488 -> 3004 0.79 of the time, 76 rows 1136 -> 3417 0.86, 157
        // rows 912 -> 2447, 385 tiles, 0.85; but 96 rows 880 -> 2874, 270 tiles, 4.35 against 4.79, 612 rows 1232 -> 432 4.74 against 5.28).
        if (tiles > 256 && tiles <= (steps >= 32 ? 512 : 448) && steps >= 12)
        {
            const bool whole = p->ragged_ck == 0 && g.Ci % 64 == 0;
            if (steps >= 28 || tiles > kSmallConvMostTiles || (whole ? (g.Co + 63) / 64 * 20 <= 11 * columns : M <= 256 && (steps >= 16 || tiles >= 364))) return 1;
        }
        // Layers whose weights the persistent kernel keeps in LDS: that takes a launch 5.2 us whatever its size (28 x 28 x 128 -> 512, one image
        // 5.23 -> 3.48, two 5.30 -> 3.79; 40 x 40 x 96 -> 288 5.52 -> 3.62); over 64 channels it takes 3.80 against 3.71 here, over 32 3.77 against 3.80.
        return p->pw_bn != 0 && !p->pw_forced && g.Ci > 64 && tiles > kSmallConvMostTiles && tiles <= 1024 ? 7 : -1;
    }
    const int forced = p->tile_override > 5000 ? p->tile_override - 5001 : -1;
    if (p->tile_override == 0)
    {
        // Few rows (small_conv_kernel.h): the panel pays where taps are whole k-steps and many.  One image unless said: 14 x 14 x 256 5.26 -> 4.40
        // us, 7 x 7 x 512 7.26 -> 5.40, 28 x 28 x 128 4.27 -> 4.03, eight images 14 x 14 x 256 7.66 -> 5.0, 5 x 5 over 9 x 9 x 384, 20 images, 12.2 -> 8.2; but 56 x
        // 56 x 64 3.37 against 3.85, and taps that are no whole k-steps 0.85 to 0.95 of the rate.  At stride 2 the panel has four times
        // the pixels: from 512 channels on (7.60 -> 7.20; 256 5.35 against 5.40, 128 4.54 against 4.80).
        // It has to serve nine taps or more (2 x 2 over 24 x 24 x 448 4.58 us against 5.01, 1 x 7 over 15 x 15 x 192 4.32 against 4.57), and be short beside
        // its outputs and k-steps: input pixels per output of up to nine (18 k-steps: 11 x 138 x 128 9.7 and 4.44 against 4.98, 36: 56 x 56 x 256 dilated by
        // 2 8.1 and 8.06 -> 7.11, by 4 15.2 and 8.07 against 15.2), or twelve from 63 k-steps on (46 x 46 x 192 under 5 x 5 at stride 2 10.7 and 7.9 -> 7.3, 10 x 10
        // x 320 under 32 x 1 13.8 and 9.9 against 11.4; 32 k-steps under 32 x 1 33 and 4.59 against 6.48).
        // Dilated filters from a second round of tiles on (8 x 36 x 36 x 128 under 4 x 4 7.0 -> 5.8, 39 x 39 x 192 under 5 x 5, three images, 9.4 -> 8.2; below it 18 x 18
        // x 64 under 5 x 5, four images, 4.20 against 4.72, 34 x 34 x 192 under 4 x 4 5.08 against 6.06).
        if (tiles <= kSmallConvMostTiles)
        {
            const bool pays = p->ragged_ck == 0 && g.Ci % 64 == 0 && steps >= (g.stride_x * g.stride_y == 1 ? 18 : 63) && g.Kh * g.Kw >= 9 &&
                              ((g.dil_x == 1 && g.dil_y == 1) || tiles > 256);
            return pays && TapRun(Window(g), M, 32) <= 32 * (steps >= 63 ? 12 : 9) ? 0 : -1;
        }
        // 256-row tiles of one wave per SIMD that fill the chip, where they are as wide (28 x 28 x 512, 32 images, 62.7 us here, 63.3 there, and 59
        // against 55 beside other launches) or the panel has four times the pixels, at
        // stride 2 (56 x 56 x 256 to 512 channels, 32 images, 57 us against 50, 120 x 120 x 128 to 256, eight, 17.9 against 19.2); elsewhere 80 us there are 63 here
        if (g.Ci % 128 == 0 && (Fill256Rows(p, M, 256) || (g.stride_x * g.stride_y > 1 && Fill256Rows(p, M, 128)))) return -1;
        // 64 channels at stride 1 that the kernel with weights in registers does not take (held_conv.hip): the resident-tile kernel, whose weights pass LDS, from
        // the size on where all its blocks are busy (56 x 56 to 64 channels, 32 and 64 images 9.7 and 15.4 us against 9.9 and 15.6; eight 6.0 against 5.6),
        // unless other launches share the device
        if (p->halo_ok && g.Ci == 64 && p->zw_neg == 0 && p->concurrency <= 1 && tiles >= 3136) return -1;
    }
    const Account accounts[kTapTiles] = {TileAccount<4, 32, 32>(p, M, steps), TileAccount<4, 32, 64>(p, M, steps), TileAccount<2, 64, 64>(p, M, steps), TileAccount<2, 128, 64>(p, M, steps),
                                         TileAccount<1, 128, 64>(p, M, steps), TileAccount<1, 64, 64>(p, M, steps), TileAccount<2, 64, 128>(p, M, steps), TileAccount<2, 32, 64>(p, M, steps)};
    // The shortest span; beside other launches what the launch takes from them counts as well, and the last two tiles do not pay (ResNet-50 at 32
    // images, its 14 x 14 x 256 layers on 64 x 64 tiles 373.5 us, on 32 x 64 tiles 379.6).
    const bool shared = p->concurrency > 1;
    const auto cost = [&](const Account& a) { return a.span + (shared ? 2.0 * a.work : 0.0); };
    if (forced >= 0) return forced < kTapTiles && accounts[forced].span > 0.0 ? forced : -1;
    int best = -1;
    for (int i = 0; i < (shared ? kTapTiles - 2 : kTapTiles); ++i)
        if (accounts[i].span > 0.0 && (best < 0 || cost(accounts[i]) < cost(accounts[best]))) best = i;
    // Panels of a wide stride that fill a CU's LDS by themselves, one after the other: 28 x 28 x 512 at stride 2, 64 images 85 us here and 41 on 128 x
    // 128 tiles, 16 images 27.9 and 23, eight 15.4 and 17; 112 x 112 x 256 to 64 channels, eight images, 21 and 14.
    if (best >= 0 && p->tile_override == 0 && g.stride_x * g.stride_y > 1 && accounts[best].alone_in_turns) return -1;
    // Wide rows, tall filters and wide dilations: where a good part of a block's work is to bring its run, kernels that read pixels per tap may be faster, by their
    // account (160 x 160 x 64 under 9 x 1, two images, 8.4 us against 16.3; 148 x 148 x 64 dilated by 6 7.6 against 18.2; 224 x 224 x 256 to 64 channels 19.4 against
    // 27.4, to 256 51 against 65; but 112 x 112 x 448 to 48 21.9 -> 12.4, 93 x 93 x 192 to 32, two images, 11.9 -> 6.9).  Of 342 layers above the small tiles
    // 72 took over 3 % longer here than there, up to 4.3 times; with the line four do, three of them by 5 %, one by a third, and of 330 layers that it was not drawn from
    // seven, by up to 15 %.
    if (best >= 0 && p->tile_override == 0 && accounts[best].bringing >= 0.37 && accounts[best].us > 0.95 * TiledUs(p, M)) return -1;
    return best;
}

template <int KG, int BM, int BN>
static int LaunchTile(const mi355x_conv2d_s* p, uint32_t batch, const void* x, void* y, const uint8_t* res, const AddFuse* add, hipStream_t stream)
{
    const bool aw = p->zw_neg != 0;
    if (p->ragged_ck != 0)
        return aw ? LaunchT<KG, BM, BN, true, true, false>(p, batch, x, y, res, add, stream) : LaunchT<KG, BM, BN, false, true, false>(p, batch, x, y, res, add, stream);
    if (p->geom.Ci % 64 != 0)
        return aw ? LaunchT<KG, BM, BN, true, false, false>(p, batch, x, y, res, add, stream) : LaunchT<KG, BM, BN, false, false, false>(p, batch, x, y, res, add, stream);
    return aw ? LaunchT<KG, BM, BN, true, false, true>(p, batch, x, y, res, add, stream) : LaunchT<KG, BM, BN, false, false, true>(p, batch, x, y, res, add, stream);
}

int mi355x::LaunchTapPanel(const mi355x_conv2d_s* p, int tile, uint32_t batch, const void* x, void* y, const uint8_t* res, const AddFuse* add, hipStream_t stream)
{
    switch (tile)
    {
    case 0: return LaunchTile<4, 32, 32>(p, batch, x, y, res, add, stream);
    case 1: return LaunchTile<4, 32, 64>(p, batch, x, y, res, add, stream);
    case 2: return LaunchTile<2, 64, 64>(p, batch, x, y, res, add, stream);
    case 3: return LaunchTile<2, 128, 64>(p, batch, x, y, res, add, stream);
    case 4: return LaunchTile<1, 128, 64>(p, batch, x, y, res, add, stream);
    case 5: return LaunchTile<1, 64, 64>(p, batch, x, y, res, add, stream);
    case 6: return LaunchTile<2, 64, 128>(p, batch, x, y, res, add, stream);
    default: return LaunchTile<2, 32, 64>(p, batch, x, y, res, add, stream);
    }
}
