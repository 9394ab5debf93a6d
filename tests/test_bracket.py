"""The constants of the requantization's fast path (csrc/bracket.h) on the CPU: the bracket encloses the reference's value for every
channel, and a channel that is dead, saturated or far wider than the others leaves the others' width alone."""
import os
import subprocess

import pytest

from tests.conftest import ROOT

PROGRAM = r"""
#include "bracket.h"
#include <cstdio>
#include <cstdint>
#include <cstring>
#include <random>
#include <string>
using namespace mi355x;
static float AsFloat(int32_t v) { float f; std::memcpy(&f, &v, 4); return f; }
// v_cvt_pknorm_u16_f32: rint(65535 x), saturated
static int HighByte(float x)
{
    const double v = std::nearbyint(65535.0 * static_cast<double>(x));
    return static_cast<int>(v < 0.0 ? 0.0 : v > 65535.0 ? 65535.0 : v) >> 8;
}
// the reference's code as an unsigned byte: fp32 multiply, add, divide, round half away from zero, add the offset, clamp
static int Reference(long long acc, float mult, float biasf, float scale, int offset, int bias)
{
    const float product = static_cast<float>(acc) * mult, f = product + biasf, t = std::round(f / scale);
    float v = static_cast<float>(offset) + t;
    v = std::fmax(v, bias ? -128.0f : 0.0f);
    v = std::fmin(v, bias ? 127.0f : 255.0f);
    return static_cast<int>(v) + bias;
}
struct Plan
{
    std::vector<float> mult, biasf, m, b;
    std::vector<double> most;
    float scale = 0.0235f;
    int offset = -3, bias = 128;
    double of_all = 0.0;
    Bracket k;
    explicit Plan(int n, double sums, unsigned seed)
    {
        std::mt19937 g(seed);
        std::uniform_real_distribution<double> r(0.0, 1.0);
        for (int c = 0; c < n; ++c)
        {
            mult.push_back(static_cast<float>(0.0235 * (0.002 + 0.018 * r(g))));
            biasf.push_back(static_cast<float>(std::rint((r(g) - 0.5) * 2000.0)) * mult.back());
            most.push_back(sums * (0.5 + 0.5 * r(g)));
        }
        of_all = sums;
    }
    void Choose()
    {
        m.assign(mult.size(), 0.0f); b = m;
        k = ChooseBracket(mult.data(), biasf.data(), most.data(), static_cast<int>(mult.size()), scale, offset + bias, true, of_all, m.data(), b.data());
    }
    // sums of every size, from zero and from where the code changes: a closed bracket gives the reference's code
    long long Check(double* open_share)
    {
        long long values = 0, open = 0, wrong = 0;
        for (size_t c = 0; c < mult.size(); ++c)
        {
            const long long most_c = static_cast<long long>(most[c]);
            const double at_zero = mult[c] != 0.0f ? -static_cast<double>(biasf[c]) / mult[c] : 0.0;
            std::mt19937_64 g(c);
            const bool marked = m[c] == 0.0f && HighByte(b[c]) == 128 && HighByte(b[c] - k.two_c) == 127;
            for (int i = 0; i < 3000 && !marked; ++i)
            {
                const double spread = std::ldexp(static_cast<double>(most_c) + 1.0, -static_cast<int>(g() % 24)) * (static_cast<double>(g() % 2000001) / 1e6 - 1.0);
                long long acc = std::llrint((i & 1 && std::fabs(at_zero) < most[c] ? at_zero : 0.0) + spread);
                acc = std::max(-most_c, std::min(most_c, acc));
                const float v = k.bits ? AsFloat(0x4b400000 + static_cast<int32_t>(acc)) - 12582912.0f : static_cast<float>(acc);
                const float p = std::fmaf(v, m[c], b[c]), q = p - k.two_c;
                const int hi = HighByte(p), lo = HighByte(q);
                ++values;
                if (hi != lo) { ++open; continue; }
                if (hi != Reference(acc, mult[c], biasf[c], scale, offset, bias) && ++wrong < 5)
                    std::printf("channel %zu sum %lld: %d, the reference %d\n", c, acc, hi, Reference(acc, mult[c], biasf[c], scale, offset, bias));
            }
        }
        *open_share = values ? static_cast<double>(open) / values : 0.0;
        return wrong;
    }
};
#define CHECK(c) do { if (!(c)) { std::printf("%s: line %d: %s\n", kind, __LINE__, #c); return 1; } } while (0)
int main(int, char** argv)
{
    const char* const kind = argv[1];
    for (int channels : {32, 128, 512})
        for (double sums : {1.0e5, 4.0e6, 3.0e7, 1.3e8})
        {
            Plan plain(channels, sums, 3), odd(channels, sums, 3);
            plain.Choose();
            const std::string what = kind;
            const size_t c = 5;
            if (what == "no_weights") { odd.mult[c] = 1e-40f; odd.biasf[c] = 0.1f; odd.most[c] = 0.0; }
            if (what == "smallest_scale") { odd.mult[c] = 1.2e-38f * 0.0235f; odd.biasf[c] = 0.3f; }
            if (what == "always_least") odd.biasf[c] = static_cast<float>(-1e7 * odd.scale);
            if (what == "always_most") { odd.most[c] = 1000.0; odd.biasf[c] = static_cast<float>(3e5 * odd.scale); }
            if (what == "wide") { odd.mult[c] = 0.5f; odd.biasf[c] = static_cast<float>(3e5 * odd.scale); odd.most[c] = 1.0e5; }
            if (what == "none") { odd.mult[c] = INFINITY; }
            odd.Choose();
            double share = 0.0;
            CHECK(plain.Check(&share) == 0 && share < 0.02);
            CHECK(odd.Check(&share) == 0 && share < 0.02);
            // others' width and form of the sums as without the odd channel (one and a half of it where that channel takes part)
            CHECK(odd.k.two_c <= 1.5f * plain.k.two_c);
            CHECK(odd.k.bits == plain.k.bits);
            CHECK(odd.k.all_fast == (what != "wide" && what != "none"));
            if (what == "always_least") CHECK(HighByte(odd.b[c]) == 0 && odd.m[c] == 0.0f);
            if (what == "always_most") CHECK(HighByte(odd.b[c]) == 255 && HighByte(odd.b[c] - odd.k.two_c) == 255 && odd.m[c] == 0.0f);
        }
    return 0;
}
"""


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    at = tmp_path_factory.mktemp("bracket")
    src, exe = at / "bracket.cpp", at / "bracket"
    src.write_text(PROGRAM)
    subprocess.run(["g++", "-O2", "-std=c++17", "-mfma", "-ffp-contract=off", "-Wall", "-Werror", f"-I{os.path.join(ROOT, 'armnn_amd', 'csrc')}", str(src), "-o", str(exe)],
                   check=True)
    return str(exe)


@pytest.mark.parametrize("kind", ["no_weights", "smallest_scale", "always_least", "always_most", "wide", "none"])
def test_an_odd_channel_leaves_the_others_alone(kind, program):
    r = subprocess.run([program, kind], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout
