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

// Taps, bit ky Kw + kx, that lie inside an H x W image for the output whose first tap is at (iy, ix), for filters of up to 32 taps, dy rows and dx columns
// apart: columns lo .. hi - 1 of the filter, the same in rows lo .. hi - 1.  tap_rows: bits 0, Kw, 2 Kw, ... (Kh - 1) Kw.  by_dy, by_dx: an integer up to (K + 1)
// d of the axis divided by d.
template <class DivY, class DivX>
constexpr uint32_t TapsInside(int iy, int ix, int H, int W, int Kh, int Kw, int dy, int dx, uint32_t tap_rows, DivY by_dy, DivX by_dx)
{
    // pixels 0 .. v of an axis, of the filter's at most, and one step of it less a pixel (a maximum and a minimum: with comparisons and selects launches took
    // up to 0.13 us longer, 5 x 5 over 16 x 28 x 28 x 64 10.89 -> 10.76, 3 x 3 over 16 x 14 x 14 x 256 6.40 -> 6.33)
    const auto reach = [](int v, int K, int d) { return std::min(std::max(v, 0), K * d) + d - 1; };
    const int xl = by_dx(reach(-ix, Kw, dx)), xh = by_dx(reach(W - ix, Kw, dx)), yl = by_dy(reach(-iy, Kh, dy)), yh = by_dy(reach(H - iy, Kh, dy));
    const uint32_t cols = static_cast<uint32_t>((1ull << xh) - (1ull << xl));      // (xh is 32 in a row of 32 taps)
    const uint32_t rows = tap_rows & static_cast<uint32_t>((1ull << (yh * Kw)) - (1ull << (yl * Kw)));
    return xh > xl && yh > yl ? cols * rows : 0u;
}

} // namespace mi355x
