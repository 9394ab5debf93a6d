// Launches of the register-staged implicit GEMM.
#include "igemm.h"

#include "common.h"
#include "conv_kernels.h"
#include "row_panel_kernel.h"
#include "small_conv_kernel.h"

using namespace mi355x;

namespace
{
template <int BM, int BN, int WM, int WN, int D, int BK, bool UT, bool AW, bool RG>
int LaunchIgemmT(const mi355x_conv2d_s* p, uint32_t batch, const void* x, void* y, hipStream_t stream)
{
    const ConvGeom& g = p->geom;
    IgemmArgs a;
    a.x = static_cast<const uint8_t*>(x);
    a.pad16 = p->pad16;
    a.w = p->w_mfma;
    a.ct = ChanTab{p->chan, p->Co_pad};
    a.corr = p->corr;
    a.y = static_cast<uint8_t*>(y);
    const long long M = static_cast<long long>(batch) * g.Ho * g.Wo;
    if (M > 0x7fffffffll / 2) return SetError(MI355X_ERR_UNSUPPORTED, "too many output pixels for one launch (%lld)", M);
    a.M = static_cast<int>(M);
    a.H = g.H; a.W = g.W; a.Ci = g.Ci; a.Ho = g.Ho; a.Wo = g.Wo; a.Co = g.Co;
    if (RG)
    {
        a.Ck = p->ragged_ck;
        a.x_last16 = a.x + static_cast<long long>(batch) * g.H * g.W * g.Ci - 16;     // (an image has at least 16 bytes)
    }
    a.vec_out = (g.Co & 15) == 0 && (reinterpret_cast<uintptr_t>(y) & 15) == 0;
    a.Kh = g.Kh; a.Kw = g.Kw;
    a.pad_top = g.pad_top; a.pad_left = g.pad_left; a.stride_x = g.stride_x; a.stride_y = g.stride_y;
    a.dil_x = g.dil_x; a.dil_y = g.dil_y;
    a.K_pad = p->K_pad;
    a.unit = (g.Kh == 1 && g.Kw == 1 && g.stride_x == 1 && g.stride_y == 1 && g.pad_top == 0 && g.pad_left == 0 && g.Ho == g.H &&
              g.Wo == g.W) ? 1 : 0;
    if (a.unit) { a.H = 1; a.W = a.M; a.Ho = 1; a.Wo = a.M; }      // one row of M pixels
    a.tiles_m = static_cast<int>((M + BM - 1) / BM);
    a.tiles_n = (g.Co + BN - 1) / BN;
    a.xor_mask = p->xor_mask;
    a.pad_word = p->pad_word;
    a.zw_neg = p->zw_neg;
    a.rowsum_bias = p->rowsum_bias;
    if (p->k_tail)
    {
        // K_pad is a multiple of 128 for the kernels with such k-tiles; here it need not be
        a.k_tiles = (p->K + BK - 1) / BK;
        a.rowsum_bias = (a.k_tiles * BK - p->K) * static_cast<int>(static_cast<int8_t>(p->pad_word & 0xffu));
    }
    a.rq = p->rq;
    const int nblocks = a.tiles_m * a.tiles_n;
    const int grid = (nblocks + 7) / 8 * 8;
    constexpr int smem = IgemmSmemBytes<BM, BN, BK>();
    static const hipError_t attr = hipFuncSetAttribute(reinterpret_cast<const void*>(&IgemmKernel<BM, BN, WM, WN, D, BK, UT, AW, RG>),
                                                       hipFuncAttributeMaxDynamicSharedMemorySize, smem);
    MI355X_HIP(attr);
    NoteKernel("IgemmKernel<%d, %d, %d, %d, %d, %d, %s, %s, %s>", BM, BN, WM, WN, D, BK, BoolName(UT), BoolName(AW), BoolName(RG));
    hipLaunchKernelGGL((IgemmKernel<BM, BN, WM, WN, D, BK, UT, AW, RG>), dim3(grid), dim3(256), smem, stream, a);
    MI355X_HIP(hipGetLastError());
    return 0;
}

// uniform-tap variant whenever a k-tile cannot straddle two filter taps; row sums when the weights have a zero point
template <int BM, int BN, int WM, int WN, int D, int BK>
int LaunchTile(const mi355x_conv2d_s* p, uint32_t batch, const void* x, void* y, hipStream_t stream)
{
    if constexpr (BK == 64)
    {
        if (p->ragged_ck != 0)
            return p->zw_neg != 0 ? LaunchIgemmT<BM, BN, WM, WN, D, BK, false, true, true>(p, batch, x, y, stream)
                                  : LaunchIgemmT<BM, BN, WM, WN, D, BK, false, false, true>(p, batch, x, y, stream);
    }
    const bool ut = (p->geom.Ci % BK) == 0;
    if (p->zw_neg != 0)
        return ut ? LaunchIgemmT<BM, BN, WM, WN, D, BK, true, true, false>(p, batch, x, y, stream)
                  : LaunchIgemmT<BM, BN, WM, WN, D, BK, false, true, false>(p, batch, x, y, stream);
    return ut ? LaunchIgemmT<BM, BN, WM, WN, D, BK, true, false, false>(p, batch, x, y, stream)
              : LaunchIgemmT<BM, BN, WM, WN, D, BK, false, false, false>(p, batch, x, y, stream);
}
} // namespace

int mi355x::LaunchIgemm(const mi355x_conv2d_s* p, int tile, uint32_t batch, const void* x, void* y, hipStream_t stream)
{
    const bool bk128 = p->bk128;
    if (tile == 64) return bk128 ? LaunchTile<64, 64, 2, 2, 2, 128>(p, batch, x, y, stream) : LaunchTile<64, 64, 2, 2, 2, 64>(p, batch, x, y, stream);
    if (p->geom.Co <= 64 || tile == 96)
        return bk128 ? LaunchTile<128, 64, 2, 2, 2, 128>(p, batch, x, y, stream) : LaunchTile<128, 64, 2, 2, 2, 64>(p, batch, x, y, stream);
    return bk128 ? LaunchTile<128, 128, 2, 2, 2, 128>(p, batch, x, y, stream) : LaunchTile<128, 128, 2, 2, 2, 64>(p, batch, x, y, stream);
}

int mi355x::PackFragments(const mi355x_conv2d_s* p, bool interleave, int8_t** out)
{
    const int steps = (p->geom.Kh * p->geom.Kw * (p->ragged_ck ? p->ragged_ck : p->geom.Ci) + 63) / 64;
    const long long pieces = static_cast<long long>(p->Co_pad / 16) * steps * 64;
    hipStream_t stream;
    if (const int rc = UploadStream(&stream)) return rc;
    MI355X_HIP(hipMalloc(reinterpret_cast<void**>(out), pieces * 16));
    hipLaunchKernelGGL(PackFragKernel, dim3(static_cast<unsigned>((pieces + 255) / 256)), dim3(256), 0, stream, p->w_mfma, *out, p->K_pad, steps, pieces, interleave ? 1 : 0);
    MI355X_HIP(hipGetLastError());
    MI355X_HIP(hipStreamSynchronize(stream));
    return 0;
}

int mi355x::LaunchSmallConv(const mi355x_conv2d_s* p, uint32_t batch, const void* x, void* y, const uint8_t* res, const AddFuse* add, hipStream_t stream)
{
    IgemmArgs a;
    bool unit_fast = false;
    if (const int rc = FillIgemmLdsArgs(p, 32, 32, batch, x, y, &a, &unit_fast)) return rc;
    a.vec_out = (p->geom.Co & 15) == 0 && (reinterpret_cast<uintptr_t>(y) & 15) == 0;
    a.w = p->w_frag;
    if (res) { a.res = res; a.add = *add; }
    const int grid = (a.tiles_m * a.tiles_n + 7) / 8 * 8;
    const bool aw = p->zw_neg != 0, rg = p->ragged_ck != 0;
    if (rg)
    {
        a.Ck = p->ragged_ck;
        a.x_last16 = a.x + static_cast<long long>(batch) * p->geom.H * p->geom.W * p->geom.Ci - 16;
    }
    const int tap_bytes = rg ? a.Ck : a.Ci, steps = (a.Kh * a.Kw * tap_bytes + 63) / 64;
    for (int w = 0; w <= 4; ++w)
    {
        const int step = steps * w / 4, tap = step * 64 / tap_bytes;
        a.wave_k[w] = {step, tap / a.Kw, tap % a.Kw, step * 64 % tap_bytes};
    }
    // x * ceil(2^32 / d) / 2^32 is x / d rounded down as long as x d < 2^32
    if (static_cast<long long>(a.M) * std::max(a.Wo, a.Ho) < 0x100000000ll)
    {
        a.wo_magic = static_cast<uint32_t>(0x100000000ull / a.Wo + (0x100000000ull % a.Wo != 0));
        a.ho_magic = static_cast<uint32_t>(0x100000000ull / a.Ho + (0x100000000ull % a.Ho != 0));
    }
    // (5 x 5 filters take the loop, from a graph 256 channels 9.45 -> 9.31 us, 512 16.6 -> 16.2; smaller ones the selects: small_conv_kernel.h)
    const bool whole = !rg && a.Ci % 64 == 0 && a.Kh * a.Kw <= 9;
    NoteKernel("SmallConvKernel<%s, %s, %s>", BoolName(aw), BoolName(rg), BoolName(whole));
    const auto kernel = rg      ? (aw ? SmallConvKernel<true, true, false> : SmallConvKernel<false, true, false>)
                        : whole ? (aw ? SmallConvKernel<true, false, true> : SmallConvKernel<false, false, true>)
                                : (aw ? SmallConvKernel<true, false, false> : SmallConvKernel<false, false, false>);
    hipLaunchKernelGGL(kernel, dim3(grid), dim3(256), 0, stream, a);
    MI355X_HIP(hipGetLastError());
    return 0;
}

template <int CG, int KB, bool AW>
static int LaunchRowPanelT(const mi355x_conv2d_s* p, uint32_t batch, const void* x, void* y, const uint8_t* res, const AddFuse* add, hipStream_t stream)
{
    IgemmArgs a;
    bool unit_fast = false;
    if (const int rc = FillIgemmLdsArgs(p, 64, 64 * CG, batch, x, y, &a, &unit_fast)) return rc;
    a.w = p->w_frag;
    if (res) { a.res = res; a.add = *add; }
    const long long nblocks = static_cast<long long>(a.tiles_m) * a.tiles_n;
    if (nblocks * a.tiles_n >= (1ll << 32) || nblocks > 0x7fffffffll - 8) return SetError(MI355X_ERR_UNSUPPORTED, "grid too large");
    const uint32_t rcp = static_cast<uint32_t>(((1ull << 32) + static_cast<uint32_t>(a.tiles_n) - 1) / static_cast<uint32_t>(a.tiles_n));
    const int grid = static_cast<int>((nblocks + 7) / 8 * 8);
    NoteKernel("RowPanelKernel<%d, %d, %s>", CG, KB, BoolName(AW));
    hipLaunchKernelGGL((RowPanelKernel<CG, KB, AW>), dim3(grid), dim3(256), RowPanelSmem<CG>(a.Ci), stream, a, p->Co_pad / 16, rcp);
    MI355X_HIP(hipGetLastError());
    return 0;
}

template <int CG, bool AW>
static int LaunchRowPanelK(const mi355x_conv2d_s* p, uint32_t batch, const void* x, void* y, const uint8_t* res, const AddFuse* add, hipStream_t stream)
{
    return p->geom.Ci <= 128 ? LaunchRowPanelT<CG, 128, AW>(p, batch, x, y, res, add, stream)
           : p->geom.Ci <= 256 ? LaunchRowPanelT<CG, 256, AW>(p, batch, x, y, res, add, stream)
                               : LaunchRowPanelT<CG, kRowPanelK, AW>(p, batch, x, y, res, add, stream);
}

int mi355x::LaunchRowPanel(const mi355x_conv2d_s* p, uint32_t batch, const void* x, void* y, const uint8_t* res, const AddFuse* add, hipStream_t stream)
{
    const bool aw = p->zw_neg != 0;
    if (p->geom.Co <= 64) return aw ? LaunchRowPanelK<1, true>(p, batch, x, y, res, add, stream) : LaunchRowPanelK<1, false>(p, batch, x, y, res, add, stream);
    return aw ? LaunchRowPanelK<2, true>(p, batch, x, y, res, add, stream) : LaunchRowPanelK<2, false>(p, batch, x, y, res, add, stream);
}
