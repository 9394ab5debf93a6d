// The constants of the requantization's fast path (device_math.h tells what the bracket is), chosen on the host.
#pragma once

#include <algorithm>
#include <cmath>
#include <vector>

namespace mi355x
{

struct Bracket
{
    float two_c;       // its width, one for the plan
    bool  all_fast;    // every channel has a fast path
    bool  bits;        // the bits of a raised accumulator may stand for the sum
};

// m, b and what follows for the plan, from `n` channels' mult and biasf and the most that the magnitude of a channel's sum can be.
// `offset`: of the output, as the codes are unsigned bytes; `allowed`: the output's scale and offset permit a fast path at all.
//   The width is the widest channel's, so that it costs a kernel one number.  A channel can therefore make every channel's values be
// settled one by one more often, and the rules keep that to channels whose values really are that uncertain:
//   - One that is saturated whatever its sum, as a pruned channel with a large bias is, gets a constant code and asks for nothing.
//   - One whose product of scales is so small that m would be subnormal (an all-zero channel's scale is often the smallest
//     float) gets m = 0; what its sums could add to the bias is part of its width.
//   - One that is wider than the others by so much that it would have more of their values settled than it has itself is left without a
//     fast path.
// One odd channel, us a launch (64 images; in brackets with the widest channel's width and none of these rules), channels without weights or with
// the smallest scale, always saturated, with biases of 1000, 4000 and 20000 codes that some sums take back:
//   1x1 128 -> 128, 56 x 56          13.8    13.8 (16.3)    13.9 (16.2)    14.2 (13.9)    14.9 (14.5)    16.2 (16.0)
//   3x3 64 -> 64, 56 x 56            14.9    14.8 (16.4)    14.8 (16.2)    15.3 (15.2)    15.5 (15.7)    16.4 (16.4)
//   depthwise 3x3, 112 x 112 x 32    14.7    14.7 (19.7)    14.6 (19.5)    (sums of nine products take back no such bias)
// A bias of 20000 codes, eighty times the type's range, is what the one width still costs: a width per channel would cost every kernel a
// register or an FMA per value.
inline Bracket ChooseBracket(const float* mult, const float* biasf, const double* most, int n, float scale, double offset, bool allowed,
                             double most_of_all, float* m, float* b)
{
    constexpr double u = 1.0 / 16777216.0;            // unit roundoff of fp32
    constexpr double unit = 256.0 / 65535.0;          // a code on the scale of m and b
    constexpr double whole = 1 << 22;                 // 1.5 * 2^23 + sum steps in ones up to here
    const double s_out = scale;
    // (SettleDev: nothing near the ends of fp32)
    allowed = allowed && s_out > 0x1p-90 && s_out < 0x1p90;
    // |t - offset| of a value that is not saturated
    const double most_t = std::max(std::fabs(257.5 - offset), std::fabs(-1.5 - offset));
    struct Line { double slope, at_zero, width; bool fast; };        // in codes
    std::vector<Line> lines(n);
    std::vector<double> widths;
    for (int c = 0; c < n; ++c)
    {
        const double fm = static_cast<double>(mult[c]) / s_out, fb = static_cast<double>(biasf[c]) / s_out, bias = std::fabs(fb);
        const double sums = most[c] * std::fabs(fm), margin = 1.0 + 8.0 * u * (sums + bias);
        Line& l = lines[c];
        l = Line{fm, fb + offset, 0.0, false};
        if (!allowed || !std::isfinite(fm) || !std::isfinite(fb) || sums >= 268435456.0) continue;
        l.fast = true;
        if (l.at_zero + sums < -margin || l.at_zero - sums > 255.0 + margin)
        {
            l.at_zero = l.at_zero < 0.0 ? 0.0 : 255.0;
            l.slope = 0.0;
            continue;
        }
        // Half-width in codes: the reference multiplies, adds the bias and divides, on values of up to |t| + |bias|, |t| and |t| codes (1.02
        // for the second order); both sides convert the sum, which rounds from 2^24 on; m and b are off by what they are off; p and
        // q round on a scale where 256 codes are 1 (128 each).
        const double slope = fm * unit, at_zero = (256.0 * (fb + offset + 0.5) - 0.5) / 65535.0, reach = most_t + bias;
        const bool normal = std::isnormal(static_cast<float>(slope));
        const double slope_off = normal ? std::fabs(static_cast<double>(static_cast<float>(slope)) / slope - 1.0) * reach : sums;
        if (!normal) l.slope = 0.0;
        l.width = u * (1.02 * (reach + 2.0 * most_t) + (most[c] >= 16777216.0 && reach >= 16777216.0 * std::fabs(fm) ? 2.04 * reach : 0.0) + 256.0) + slope_off +
                  0.5 * std::ldexp(1.0, std::ilogb(std::fabs(at_zero) + 0.001) - 23) / unit;
        l.fast = l.width < 0.0625;
        if (l.fast) widths.push_back(l.width);
    }
    // the width that leaves the fewest values to be settled
    std::sort(widths.begin(), widths.end());
    double c_codes = 1024.0 * u, least = static_cast<double>(widths.size());         // (1024 u: enough to tell p from q anywhere)
    for (size_t i = 0; i < widths.size(); ++i)
    {
        const double c = std::max(1024.0 * u, widths[i]), settled = 2.0 * c * static_cast<double>(i + 1) + static_cast<double>(widths.size() - i - 1);
        if (settled > least) continue;
        least = settled;
        c_codes = c;
    }
    const double c_x = c_codes * unit;
    Bracket out;
    out.two_c = std::nextafterf(static_cast<float>(2.0 * c_x), 1.0f);
    out.all_fast = true;
    out.bits = most_of_all < 536870912.0;
    for (int c = 0; c < n; ++c)
    {
        const Line& l = lines[c];
        const bool fast = l.fast && l.width <= c_codes;
        // (a channel without a fast path: a byte's edge whatever the sum, p gives 128 and q 127)
        const double code = fast ? l.at_zero + 0.5 : 128.0;
        m[c] = fast ? static_cast<float>(l.slope * unit) : 0.0f;
        b[c] = static_cast<float>((256.0 * code - 0.5) / 65535.0 + c_x);
        out.all_fast &= fast;
        // where the steps are not ones, codes must be saturated
        if (m[c] != 0.0f && most[c] > whole && whole * std::fabs(l.slope) - std::fabs(l.at_zero) < 300.0) out.bits = false;
    }
    return out;
}

} // namespace mi355x
