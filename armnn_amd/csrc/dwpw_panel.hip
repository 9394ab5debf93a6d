// Launches of the fused depthwise + pointwise kernel that keeps the layer between them in LDS.
#include "dwpw_panel.h"

#include <algorithm>

#include "common.h"
#include "dwpw_panel_kernel.h"
#include "igemm.h"

using namespace mi355x;

namespace
{
template <int S, int TH, int TW, int NW, int CG, int KS, bool U>
int LaunchT(const mi355x_conv2d_s* dw, const mi355x_conv2d_s* pw, uint32_t batch, const void* x, void* y, hipStream_t stream)
{
    using G = DwPwPanelGeom<S, TH, TW, NW, CG>;
    const ConvGeom& g = dw->geom;
    const auto rcp = [](int d) { return static_cast<uint32_t>(((1ull << 32) + static_cast<uint32_t>(d) - 1) / static_cast<uint32_t>(d)); };
    DwPwPanelArgs a;
    a.x = static_cast<const uint8_t*>(x); a.pad16 = dw->pad16; a.dw_blk = dw->dw_blk.load(std::memory_order_acquire);
    a.H = g.H; a.W = g.W; a.C = g.Co; a.Ho = g.Ho; a.Wo = g.Wo;
    a.pad_top = g.pad_top; a.pad_left = g.pad_left;
    a.tiles_x = (g.Wo + TW - 1) / TW; a.tiles_y = (g.Ho + TH - 1) / TH;
    a.Co = pw->geom.Co;
    a.nb = (a.Co + G::NCOL - 1) / G::NCOL;
    const long long items = static_cast<long long>(batch) * a.tiles_x * a.tiles_y * a.nb;
    // (the divisions by reciprocals are exact while item x divisor stays below 2^32)
    if (items * std::max(a.nb, std::max(a.tiles_x, a.tiles_y)) >= (1ll << 32) || items > 0x7fffffffll - 8)
        return SetError(MI355X_ERR_UNSUPPORTED, "grid too large");
    a.total_items = static_cast<int>(items); a.xcd_chunk = static_cast<int>((items + 7) / 8);
    a.rcp_tiles_x = rcp(a.tiles_x); a.rcp_tiles_y = rcp(a.tiles_y); a.rcp_nb = rcp(a.nb); a.rcp_ng = rcp(a.C / 16);
    a.dw_xor = dw->xor_mask; a.dw_rq = dw->rq;
    a.w = pw->w_panel.load(std::memory_order_acquire); a.co_groups = pw->Co_pad / 16;
    a.pw_ct = ChanTab{pw->chan, pw->Co_pad}; a.pw_corr = pw->corr;
    a.y = static_cast<uint8_t*>(y);
    a.y_bytes = static_cast<long long>(batch) * g.Ho * g.Wo * a.Co;
    a.zw_neg = pw->zw_neg; a.mid_xor = pw->xor_mask; a.pw_rq = pw->rq;
    const int smem = G::Smem(a.C, U);
    static const hipError_t attr = hipFuncSetAttribute(reinterpret_cast<const void*>(&DwPwPanelKernel<S, TH, TW, NW, CG, KS, U>),
                                                       hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
    MI355X_HIP(attr);
    NoteKernel("DwPwPanelKernel<%d, %d, %d, %d, %d, %d, %s>", S, TH, TW, NW, CG, KS, BoolName(U));
    hipLaunchKernelGGL((DwPwPanelKernel<S, TH, TW, NW, CG, KS, U>), dim3(static_cast<unsigned>(a.xcd_chunk) * 8u), dim3(64 * NW), smem, stream, a);
    MI355X_HIP(hipGetLastError());
    return 0;
}

template <bool U, int TH, int TW, int NW, int CG, int KS>
int LaunchS(const mi355x_conv2d_s* dw, const mi355x_conv2d_s* pw, uint32_t batch, const void* x, void* y, hipStream_t stream)
{
    return dw->d.stride_x == 1 ? LaunchT<1, TH, TW, NW, CG, KS, U>(dw, pw, batch, x, y, stream)
                               : LaunchT<2, TH, TW, NW, CG, KS, U>(dw, pw, batch, x, y, stream);
}

template <bool U>
int LaunchU(const mi355x_conv2d_s* dw, const mi355x_conv2d_s* pw, uint32_t batch, const void* x, void* y, hipStream_t stream)
{
    const int C = dw->geom.Co, Co = pw->geom.Co, steps = (C + 63) / 64;
    const bool s1 = dw->d.stride_x == 1;
    const auto blocks = [&](int th, int tw, int ncol) {
        return static_cast<long long>(batch) * ((dw->geom.Wo + tw - 1) / tw) * ((dw->geom.Ho + th - 1) / th) * ((Co + ncol - 1) / ncol);
    };
    // The largest tile that still gives about 100 blocks: the depthwise layer is computed once per block of output channels and the
    // halo read again, so small tiles cost work; below that the chip idles (MobileNetV1, three passes side by side, 8 images: 54 us
    // with this line at 100, 57 at 50, 67 at 130, where 4 x 4 tiles take over).  The 8 x 8 tile of 512 output channels fills a CU's
    // registers by itself and waits for about one block per CU (32 images, alone: 9.4 us on 4 x 8 tiles, 11.6 on 8 x 8).
    // Up to 128 channels there are one or two blocks of 64 to compute: fewer waves, which share them.
    if (steps == 1 && blocks(8, 16, 128) >= 100)
        return Co <= 64 ? LaunchS<U, 8, 16, 4, 1, 1>(dw, pw, batch, x, y, stream) : LaunchS<U, 8, 16, 4, 2, 1>(dw, pw, batch, x, y, stream);
    if (steps == 2 && blocks(8, 8, 256) >= 100)
        return Co <= 128 ? LaunchS<U, 8, 8, 4, 2, 2>(dw, pw, batch, x, y, stream) : LaunchS<U, 8, 8, 4, 4, 2>(dw, pw, batch, x, y, stream);
    if ((steps == 8 || steps == 4) && Co > 256)
    {
        if (s1 && blocks(8, 8, 512) >= 200) return steps == 8 ? LaunchT<1, 8, 8, 8, 4, 8, U>(dw, pw, batch, x, y, stream) : LaunchT<1, 8, 8, 8, 4, 4, U>(dw, pw, batch, x, y, stream);
        if (blocks(4, 8, 512) >= 100) return steps == 8 ? LaunchS<U, 4, 8, 8, 4, 8>(dw, pw, batch, x, y, stream) : LaunchS<U, 4, 8, 8, 4, 4>(dw, pw, batch, x, y, stream);
    }
    if (steps == 4 && s1 && Co <= 256 && blocks(8, 8, 256) >= 200) return LaunchT<1, 8, 8, 8, 2, 4, U>(dw, pw, batch, x, y, stream);
    if (blocks(4, 8, 256) >= 100)
        return steps == 8 ? LaunchS<U, 4, 8, 8, 2, 8>(dw, pw, batch, x, y, stream) : steps == 4 ? LaunchS<U, 4, 8, 8, 2, 4>(dw, pw, batch, x, y, stream)
                                                                                              : LaunchS<U, 4, 8, 8, 2, 0>(dw, pw, batch, x, y, stream);
    if (blocks(4, 4, 256) >= 100) return LaunchS<U, 4, 4, 16, 1, 0>(dw, pw, batch, x, y, stream);
    return LaunchS<U, 4, 4, 8, 1, 0>(dw, pw, batch, x, y, stream);
}
} // namespace

bool mi355x::DwPwPanelTakes(const mi355x_conv2d_s* dw, const mi355x_conv2d_s* pw)
{
    const mi355x_conv2d_desc& a = dw->d;
    if (dw->algo != MI355X_ALGO_DEPTHWISE || dw->variant != 1 || a.out_c != a.in_c || (a.out_c & 15) != 0) return false;
    const ConvGeom& g = pw->geom;
    const bool unit = g.Kh == 1 && g.Kw == 1 && g.stride_x == 1 && g.stride_y == 1 && g.Ho == g.H && g.Wo == g.W && g.H * g.W > 1;
    if (!pw->w_mfma || !unit || pw->ragged_ck != 0 || g.Ci > 1024 || (g.Co & 15) != 0 || g.Ci != static_cast<int>(a.out_c)) return false;
    if (static_cast<long long>(a.in_h) * a.in_w * a.in_c >= (1ll << 31)) return false;
    const int smem = a.stride_x == 1 ? DwPwPanelGeom<1, 4, 8, 8, 2>::Smem(static_cast<int>(a.out_c), true) : DwPwPanelGeom<2, 4, 8, 8, 2>::Smem(static_cast<int>(a.out_c), true);
    return smem <= 160 * 1024;
}

namespace
{
// Blocks of 64 channels: kDwBlkRows rows of [16][4] dwords, entry [j][e] for channel 16 e + j of the block: corr, m, b, mult, biasf, filter taps
// 0..3, 4..7, 8, and those of the second halves.  Channels past the last one are all zero: a bracket that closes, some code that no
// weight and no row sum counts.  `grp`, `chan`, `second`: the plan's dw_grp, chan
// and w_dot4b (or null).
__global__ __launch_bounds__(256) void PackDwBlkKernel(const uint32_t* __restrict__ grp, const float* __restrict__ chan, int stride, const uint32_t* __restrict__ second, uint32_t* __restrict__ blk, int C, int dwords)
{
    const int i = static_cast<int>(blockIdx.x) * 256 + static_cast<int>(threadIdx.x);
    if (i >= dwords) return;
    const int b = i / (kDwBlkRows * 64), row = i % (kDwBlkRows * 64) / 64, c = b * 64 + i % 4 * 16 + i % 64 / 4;
    uint32_t v = 0;
    if (c < C)
    {
        const uint32_t* const of = grp + (c / 4) * kDwGrpDwords + c % 4;         // rows of four: weights 0 .. 2, corr, m, b
        if (row < 3) v = of[(3 + row) * 4];
        else if (row < 5) v = __builtin_bit_cast(uint32_t, chan[(row - 3) * stride + c]);
        else
            for (int t = (row - (row < 8 ? 5 : 8)) * 4, n = 0; n < 4 && t < 9; ++t, ++n)
            {
                const uint32_t taps = row < 8 ? of[t / 3 * 4] : second ? second[c * 4 + t / 3] : 0u;
                v |= (taps >> (8 * (t % 3)) & 0xffu) << (8 * n);
            }
    }
    blk[i] = v;
}

int PackDwBlk(const mi355x_conv2d_s* dw, uint32_t** out)
{
    const int C = dw->geom.Co, dwords = (C + 63) / 64 * (kDwBlkRows * 64);
    hipStream_t stream;
    if (const int rc = UploadStream(&stream)) return rc;
    MI355X_HIP(hipMalloc(reinterpret_cast<void**>(out), static_cast<size_t>(dwords) * 4));
    hipLaunchKernelGGL(PackDwBlkKernel, dim3(static_cast<unsigned>((dwords + 255) / 256)), dim3(256), 0, stream, dw->dw_grp, dw->chan, dw->Co_pad, dw->w_dot4b, *out, C, dwords);
    MI355X_HIP(hipGetLastError());
    MI355X_HIP(hipStreamSynchronize(stream));
    return 0;
}

// While one is open, the thread may allocate and wait although it captures a graph.
struct OutsideCapture
{
    hipStreamCaptureMode mode = hipStreamCaptureModeRelaxed;
    OutsideCapture() { (void)hipThreadExchangeStreamCaptureMode(&mode); }
    ~OutsideCapture() { (void)hipThreadExchangeStreamCaptureMode(&mode); }
};
} // namespace

int mi355x::PrepareDwPwPanel(const mi355x_conv2d_s* dw, const mi355x_conv2d_s* pw)
{
    if (dw->dw_blk.load(std::memory_order_acquire) && pw->w_panel.load(std::memory_order_acquire)) return 0;
    OutsideCapture outside;
    UploadScope uploads;
    {
        std::lock_guard<std::mutex> lock(dw->panel_mutex);
        if (!dw->dw_blk.load(std::memory_order_relaxed))
        {
            uint32_t* blk = nullptr;
            if (const int rc = PackDwBlk(dw, &blk)) { (void)hipFree(blk); return rc; }
            dw->dw_blk.store(blk, std::memory_order_release);
        }
    }
    std::lock_guard<std::mutex> lock(pw->panel_mutex);
    if (!pw->w_panel.load(std::memory_order_relaxed))
    {
        int8_t* w = nullptr;
        if (const int rc = PackFragments(pw, true, &w)) { (void)hipFree(w); return rc; }
        pw->w_panel.store(w, std::memory_order_release);
    }
    return 0;
}

int mi355x::LaunchDwPwPanel(const mi355x_conv2d_s* dw, const mi355x_conv2d_s* pw, uint32_t batch, const void* x, void* y, hipStream_t stream)
{
    return dw->w_dot4b != nullptr || pw->zw_neg != 0 ? LaunchU<true>(dw, pw, batch, x, y, stream) : LaunchU<false>(dw, pw, batch, x, y, stream);
}
