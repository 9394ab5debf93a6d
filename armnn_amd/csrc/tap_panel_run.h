// Which input pixels the blocks of TapPanelBlock (tap_panel_kernel.h) hold.
#pragma once

#include <algorithm>
#include <cstdint>

namespace mi355x
{

struct TapWindow
{
    int H, W, Ho, Wo, Kh, Kw, stride_y, stride_x, dil_y, dil_x;
};

// Output pixels are numbered through rows and images, input pixels likewise.  Whether the numbers of the pixels' first taps (padding is counted
// as if its pixels were there) rise with the outputs': then what any tap of a run of outputs reads inside its image lies between the first
// tap of the first and the last tap of the last one.
inline bool TapsInOrder(const TapWindow& w) { return (w.Ho - 1) * w.stride_y < w.H && (w.Wo - 1) * w.stride_x < w.W; }

// The most input pixels between those two taps for any `pixels` outputs of `all`.  The first tap moves by stride_x within a row; at its end by
// stride_y rows less the outputs' width, at the end of an image by the rows that no first tap stands in besides.
inline long long TapRun(const TapWindow& w, long long all, int pixels)
{
    const long long last = std::min<long long>(pixels, all) - 1, image = static_cast<long long>(w.Ho) * w.Wo;
    return w.stride_x * last + (last + w.Wo - 1) / w.Wo * std::max(0, w.stride_y * w.W - w.stride_x * w.Wo) +
           (last + image - 1) / image * std::max(0, w.H - w.Ho * w.stride_y) * w.W + static_cast<long long>(w.Kh - 1) * w.dil_y * w.W +
           static_cast<long long>(w.Kw - 1) * w.dil_x + 1;
}

// What is read for piece i of a run whose pieces lo .. hi lie inside the tensor: itself, or one of those.  A run of outputs that have all taps in the padding
// above the first image ends ahead of the tensor (hi < lo); then the tensor's first piece, lo.
constexpr int PieceInside(int i, int lo, int hi)
{
    const int upper = i < hi ? i : hi;
    return upper > lo ? upper : lo;
}

// Taps, bit ky Kw + kx, that lie inside an H x W image for the output whose first tap is at (iy, ix), for filters of up to 32 taps without dilation:
// columns lo .. hi - 1 of the filter, the same in rows lo .. hi - 1.  tap_rows: bits 0, Kw, 2 Kw, ... (Kh - 1) Kw.
constexpr uint32_t TapsInside(int iy, int ix, int H, int W, int Kh, int Kw, uint32_t tap_rows)
{
    const auto within = [](int v, int most) { return v < 0 ? 0 : v < most ? v : most; };
    const int xl = within(-ix, Kw), xh = within(W - ix, Kw), yl = within(-iy, Kh), yh = within(H - iy, Kh);
    const uint32_t cols = static_cast<uint32_t>((1ull << xh) - (1ull << xl));      // (xh is 32 in a row of 32 taps)
    const uint32_t rows = tap_rows & static_cast<uint32_t>((1ull << (yh * Kw)) - (1ull << (yl * Kw)));
    return xh > xl && yh > yl ? cols * rows : 0u;
}

} // namespace mi355x
