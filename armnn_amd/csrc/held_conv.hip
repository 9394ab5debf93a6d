#include "held_conv.h"

#include <algorithm>

#include "common.h"
#include "held_conv_kernel.h"
#include "igemm.h"
#include "tap_panel_run.h"

using namespace mi355x;

namespace
{
constexpr int kWaves = 4, kSlots = 512, kFewPieces = 4, kMostPieces = 10, kBlockLds = 80 * 1024;
using Geom = HeldConvGeom<kWaves>;

TapWindow Window(const ConvGeom& g) { return {g.H, g.W, g.Ho, g.Wo, g.Kh, g.Kw, g.stride_y, g.stride_x, g.dil_y, g.dil_x}; }

// Bytes per 16 channels of the panel for `groups` x 16 outputs
long long Pitch(const ConvGeom& g, long long M, int groups) { return ((TapRun(Window(g), M, groups * 16) + 1) | 1) * 16; }

bool Fits(const ConvGeom& g, long long M, int groups)
{
    const long long gp = Pitch(g, M, groups);
    return gp / 16 * 4 <= kMostPieces * Geom::NT && Geom::Smem(static_cast<int>(gp), groups) <= kBlockLds;
}

// Groups of 16 outputs of a block: whole rounds of two blocks per CU, as few as hold their runs in registers on the way to LDS
int GroupsOfBlock(const mi355x_conv2d_s* p, long long M)
{
    const ConvGeom& g = p->geom;
    const long long groups = (M + 15) / 16, slots = std::max(1, kSlots / ((g.Co + 63) / 64));
    for (long long rounds = 1;; ++rounds)
    {
        const int each = static_cast<int>(std::min<long long>((groups + slots * rounds - 1) / (slots * rounds), 1024));
        if (each == 1 || Fits(g, M, each)) return each;
    }
}

// Whether the kernel can run the launch
bool Takes(const mi355x_conv2d_s* p, uint32_t batch)
{
    const ConvGeom& g = p->geom;
    const long long M = static_cast<long long>(batch) * g.Ho * g.Wo, in_pixels = static_cast<long long>(batch) * g.H * g.W;
    // (pixels are decoded with reciprocals, and a pixel's number in a run stands above its taps' bits)
    return p->w_frag && HeldConvTakes(p) && M <= (1ll << 27) && in_pixels <= (1ll << 27) && M * std::max(g.Wo, g.Ho) < (1ll << 32) &&
           (M + 15) / 16 * ((g.Co + 63) / 64) * ((g.Co + 63) / 64) < (1ll << 31) && Fits(g, M, 1);
}

// ... and whether it is the fastest, its blocks working on `groups`
bool Pays(const mi355x_conv2d_s* p, uint32_t batch, int groups)
{
    const ConvGeom& g = p->geom;
    // At stride 2 and more a block's run is mostly pixels that its neighbours read as well: 64 x 112 x 112 to 64 channels 26.0 us against 24.1 on other
    // tiles, 64 x 28 x 28 to 512 11.8 against 11.1, 60 x 40 x 40 5.85 against 5.67.  Beside other launches the networks at hand gain nothing (ResNet-50,
    // 32 images in two lanes, 378 against 377 us a pass): blocks with all registers of a CU leave no room to neighbours.
    if (g.stride_x * g.stride_y > 1 || p->concurrency > 1) return false;
    // Each wave first fetches 36 KB of weights, so few outputs are better off with kernels that stream them; the longer the run, the later a
    // block starts.  Tiles of one pixel x 64 channels: 12.8 k 5.35 us against 5.05 and 5.19 against 4.66, 18.0 k 5.27 against 5.30, 18.8 k 5.28 against 5.80,
    // 23.1 k 5.34 against 5.39; with long runs 25.1 k 5.84 against 5.78, 40.0 k 6.57 against 6.92.
    const long long M = static_cast<long long>(batch) * g.Ho * g.Wo, tiles = M * ((g.Co + 63) / 64);
    if (tiles < 18000) return false;
    if (tiles < 32000 && Pitch(g, M, groups) / 16 * 4 > kFewPieces * Geom::NT) return false;
    // Wide rows, tall filters and wide dilations leave a block few outputs beside the pixels that their other taps read, and a launch rounds of blocks
    // that each fetch both the run and the weights.  A launch of one round stays ahead (one image of 224 x 224, 5.0 pixels of a run per output, 7.3 us against 8.5, 2
    // of 94 x 94 dilated by 2, 5.8 pixels, 6.8 against 7.5).  In several it does up to five pixels per output (3 images of 208 x 208, 4.3 pixels, 12.5 against 16.3, of
    // 240 x 240, 4.8 pixels, 17.4 against 18.3, of 256 x 256, 6.4 pixels, 22.1 against 18.7; 300 x 300, 19.8 pixels, 23.9 against 10.4), to over 128 channels, whose tiles
    // of 64 each fetch the run, up to four (224 x 224 to 192 channels, 3.8 pixels, 14.4 against 14.8; to 256, 4.1 pixels, 19.7 against 15.4).
    const long long slots = std::max(1, kSlots / ((g.Co + 63) / 64));
    return groups * slots >= (M + 15) / 16 || TapRun(Window(g), M, groups * 16) <= (g.Co <= 128 ? 5 : 4) * 16 * groups;
}

template <int HS, bool BITS>
int LaunchT(const HeldConvArgs& t, int smem, hipStream_t stream)
{
    typedef void (*Kernel)(HeldConvArgs);
    const Kernel kernel = HeldConvKernel<kWaves, HS, BITS>;
    static const hipError_t attr = hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, kBlockLds);
    MI355X_HIP(attr);
    NoteKernel("HeldConvKernel<%d, %d, %s>", kWaves, HS, BoolName(BITS));
    hipLaunchKernelGGL(kernel, dim3(static_cast<unsigned>((t.blocks + 7) / 8 * 8)), dim3(Geom::NT), smem, stream, t);
    MI355X_HIP(hipGetLastError());
    return 0;
}
} // namespace

bool mi355x::HeldConvTakes(const mi355x_conv2d_s* p)
{
    const ConvGeom& g = p->geom;
    return g.Ci == 64 && g.Kh * g.Kw == kHeldTaps && (g.Co & 15) == 0 && p->zw_neg == 0 && TapsInOrder(Window(g));
}

int mi355x::HeldConvGroups(const mi355x_conv2d_s* p, uint32_t batch)
{
    if ((p->tile_override != 0 && p->tile_override != 5009) || !Takes(p, batch)) return 0;
    const int groups = GroupsOfBlock(p, static_cast<long long>(batch) * p->geom.Ho * p->geom.Wo);
    return p->tile_override == 5009 || Pays(p, batch, groups) ? groups : 0;
}

int mi355x::LaunchHeldConv(const mi355x_conv2d_s* p, int groups, uint32_t batch, const void* x, void* y, hipStream_t stream)
{
    const ConvGeom& g = p->geom;
    HeldConvArgs t;
    bool unit_fast = false;
    if (const int rc = FillIgemmLdsArgs(p, 64, 64, batch, x, y, &t.g, &unit_fast)) return rc;
    t.g.w = p->w_frag;
    const auto reciprocal = [](int d) { return static_cast<uint32_t>((0x100000000ull + static_cast<uint32_t>(d) - 1) / static_cast<uint32_t>(d)); };
    t.g.wo_magic = reciprocal(g.Wo);
    t.g.ho_magic = reciprocal(g.Ho);
    t.rcp_tiles_n = reciprocal(t.g.tiles_n);
    t.groups = groups;
    t.blocks = (t.g.M + 16 * t.groups - 1) / (16 * t.groups) * t.g.tiles_n;
    t.in_pixels = static_cast<int>(static_cast<long long>(batch) * g.H * g.W);
    t.gp = static_cast<int>(Pitch(g, t.g.M, t.groups));
    t.span = (g.Kh - 1) * g.dil_y * g.W + (g.Kw - 1) * g.dil_x + 1;
    for (int i = 0; i < kHeldTaps; ++i) t.tap_at[i] = (i / g.Kw * g.dil_y * g.W + i % g.Kw * g.dil_x) * 16;
    const int smem = Geom::Smem(t.gp, t.groups);
    const bool bits = t.g.rq.acc_base != 0;
    if (t.gp / 16 * 4 <= kFewPieces * Geom::NT) return bits ? LaunchT<kFewPieces, true>(t, smem, stream) : LaunchT<kFewPieces, false>(t, smem, stream);
    return bits ? LaunchT<kMostPieces, true>(t, smem, stream) : LaunchT<kMostPieces, false>(t, smem, stream);
}
