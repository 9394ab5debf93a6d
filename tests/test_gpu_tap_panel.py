"""Convolutions whose blocks hold the run of input pixels that their taps read (csrc/tap_panel_kernel.h): how long that run can get, on the CPU; every
tile at its edges against the plain kernel, bit for bit."""
import os
import subprocess

import numpy as np
import pytest

from armnn_amd import shim, synth
from armnn_amd.tensor import QTensor, TensorInfo, numpy_dtype
from tests import cases
from tests.conftest import ROOT

U8, S8 = cases.U8, cases.S8

# every output's taps inside its image lie in the run from its block's first pixel on, for blocks that start anywhere
PROGRAM = r"""
#include "tap_panel_run.h"
#include <cstdio>
#include <random>
int main()
{
    std::mt19937 rng(7);
    auto draw = [&](int lo, int hi) { return lo + static_cast<int>(rng() % static_cast<unsigned>(hi - lo + 1)); };
    int taken = 0, bad = 0, ahead = 0;
    for (int n = 0; n < 12000; ++n)
    {
        mi355x::TapWindow w{draw(1, 19), draw(1, 19), 0, 0, draw(1, 5), draw(1, 6), draw(1, 3), draw(1, 3), draw(1, 2), draw(1, 2)};
        const int top = draw(0, 4), left = draw(0, 4), images = draw(1, 5), pixels = 32 << draw(0, 2);
        w.Ho = (w.H + top + draw(0, 4) - (w.Kh - 1) * w.dil_y - 1) / w.stride_y + 1;
        w.Wo = (w.W + left + draw(0, 4) - (w.Kw - 1) * w.dil_x - 1) / w.stride_x + 1;
        if (w.Ho < 1 || w.Wo < 1 || !mi355x::TapsInOrder(w)) continue;
        ++taken;
        const int all = images * w.Ho * w.Wo;
        const long long run = mi355x::TapRun(w, all, pixels);
        auto first = [&](int m) { const int r = m / w.Wo, i = r / w.Ho; return (i * w.H + (r - i * w.Ho) * w.stride_y - top) * w.W + (m - r * w.Wo) * w.stride_x - left; };
        const int in_pixels = images * w.H * w.W;
        for (int m0 = 0; m0 < all; ++m0)
        {
            // what a block that starts here requests lies inside the tensor
            const int base = first(m0), npx = first(std::min(m0 + pixels, all) - 1) - base + (w.Kh - 1) * w.dil_y * w.W + (w.Kw - 1) * w.dil_x + 1;
            const int lo = std::max(0, -base), hi = std::min(npx, in_pixels - base) - 1;
            ahead += hi < lo;
            for (int i = 0; i < npx + 64; ++i)
            {
                const int at = base + mi355x::PieceInside(i, lo, hi);
                if (at < 0 || at >= in_pixels || (i >= lo && i <= hi && at != base + i)) ++bad;
            }
            for (int m = m0; m < all && m < m0 + pixels; ++m)
                for (int ky = 0; ky < w.Kh; ++ky)
                    for (int kx = 0; kx < w.Kw; ++kx)
                    {
                        const int r = m / w.Wo, i = r / w.Ho;
                        const int iy = (r - i * w.Ho) * w.stride_y - top + ky * w.dil_y, ix = (m - r * w.Wo) * w.stride_x - left + kx * w.dil_x;
                        if (iy < 0 || iy >= w.H || ix < 0 || ix >= w.W) continue;
                        const long long at = (static_cast<long long>(i) * w.H + iy) * w.W + ix - first(m0);
                        if (at < 0 || at >= run) ++bad;
                    }
        }
    }
    std::printf("%d windows, %d runs ahead of the tensor, %d reads outside\n", taken, ahead, bad);
    return bad != 0 || taken < 1000 || ahead == 0;
}
"""


def test_runs_hold_what_their_taps_read(tmp_path):
    src, exe = tmp_path / "run.cpp", tmp_path / "run"
    src.write_text(PROGRAM)
    subprocess.run(["g++", "-O2", "-std=c++17", "-Wall", "-Werror", f"-I{os.path.join(ROOT, 'armnn_amd', 'csrc')}", str(src), "-o", str(exe)], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout


# every filter of up to 32 taps, its window anywhere around images narrower and wider than it: each bit against the definition
MASK_PROGRAM = r"""
#include "tap_panel_run.h"
#include <cstdio>
#include <cstdlib>
// the kernel's division: a multiplication by ceil(2^32 / d)
struct Div
{
    int d, K;
    int operator()(int v) const
    {
        if (v < 0 || v > (K + 1) * d) std::abort();
        const uint32_t rcp = static_cast<uint32_t>((0x100000000ull + d - 1) / d);
        return d == 1 ? v : static_cast<int>(static_cast<uint64_t>(v) * rcp >> 32);
    }
};
int main()
{
    long windows = 0, bad = 0;
    for (int Kh = 1; Kh <= 32; ++Kh)
        for (int Kw = 1; Kh * Kw <= 32; ++Kw)
        {
            uint32_t tap_rows = 0;
            for (int ky = 0; ky < Kh; ++ky) tap_rows |= 1u << (ky * Kw);
            for (int H : {1, 2, 5, 33, 40})
                for (int W : {1, 3, 7, 31, 32, 33, 64})
                    for (int d : {1, 2, 3, 7})
                    {
                        const int dy = d, dx = d == 3 ? 2 : d;
                        for (int iy = -(Kh - 1) * dy - 2; iy <= H + 1; iy += H < 33 || iy % 5 ? 1 : 2)
                            for (int ix = -(Kw - 1) * dx - 2; ix <= W + 1; ++ix)
                            {
                                uint32_t want = 0;
                                for (int ky = 0; ky < Kh; ++ky)
                                    for (int kx = 0; kx < Kw; ++kx)
                                        if (iy + ky * dy >= 0 && iy + ky * dy < H && ix + kx * dx >= 0 && ix + kx * dx < W) want |= 1u << (ky * Kw + kx);
                                bad += mi355x::TapsInside(iy, ix, H, W, Kh, Kw, dy, dx, tap_rows, Div{dy, Kh}, Div{dx, Kw}) != want;
                                ++windows;
                            }
                    }
        }
    std::printf("%ld windows, %ld wrong masks\n", windows, bad);
    return bad != 0;
}
"""


def test_masks_of_the_taps_inside_an_image(tmp_path):
    src, exe = tmp_path / "mask.cpp", tmp_path / "mask"
    src.write_text(MASK_PROGRAM)
    subprocess.run(["g++", "-O2", "-std=c++17", "-fsanitize=shift", "-fno-sanitize-recover=shift", "-Wall", "-Werror",
                    f"-I{os.path.join(ROOT, 'armnn_amd', 'csrc')}", str(src), "-o", str(exe)], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout + r.stderr


LAYERS = [
    ("one_pixel_c64", dict(n=1, h=1, w=1, ci=64, co=16)),
    ("31_pixels_c80_co33", dict(n=1, h=1, w=31, ci=80, co=33)),
    ("65_pixels_c64_two_columns", dict(n=5, h=1, w=13, ci=64, co=130)),
    ("images_of_9_pixels_c128", dict(n=15, h=3, w=3, ci=128, co=64)),
    ("129_pixels_c192_valid_5x5", dict(n=1, h=7, w=47, ci=192, co=48, kh=5, kw=5, padding="valid")),
    ("stride2_odd_c64", dict(n=3, h=15, w=9, ci=64, co=72, stride=(2, 2))),
    ("stride_1_2_c48", dict(n=2, h=9, w=14, ci=48, co=40, stride=(1, 2))),
    ("dilated_c112_5x5", dict(n=2, h=13, w=9, ci=112, co=36, kh=5, kw=5, dilation=(2, 1))),
    ("padding_all_round_c64", dict(n=2, h=6, w=7, ci=64, co=32, padding=(2, 0, 1, 0))),
    ("ragged_c72_stride2", dict(n=2, h=11, w=11, ci=72, co=120, stride=(2, 2))),
    ("ragged_c50_to_the_end", dict(n=1, h=8, w=9, ci=50, co=17)),
    ("filter_1x7_c80", dict(n=2, h=5, w=12, ci=80, co=64, kh=1, kw=7)),
    ("first_row_in_the_padding_c192", dict(n=1, h=9, w=200, ci=192, co=32, kh=1, kw=3, stride=(2, 2), padding=(1, 0, 1, 1))),
    ("first_row_in_the_padding_ragged_c200", dict(n=1, h=9, w=200, ci=200, co=17, kh=1, kw=3, stride=(2, 2), padding=(1, 0, 1, 1))),
    ("32_taps_in_a_row_c64", dict(n=2, h=3, w=70, ci=64, co=32, kh=1, kw=32)),
    ("32_taps_in_a_row_ragged_c72", dict(n=1, h=2, w=45, ci=72, co=17, kh=1, kw=32)),
    ("32_taps_in_a_column_c80", dict(n=1, h=40, w=3, ci=80, co=32, kh=32, kw=1)),
    ("filter_4x8_c64", dict(n=2, h=9, w=11, ci=64, co=48, kh=4, kw=8)),
    ("one_tap_c64", dict(n=3, h=7, w=5, ci=64, co=130, kh=1, kw=1)),
    ("one_tap_c1040", dict(n=65, h=1, w=1, ci=1040, co=33, kh=1, kw=1)),
    ("one_tap_ragged_c50", dict(n=1, h=3, w=43, ci=50, co=17, kh=1, kw=1)),
]


@pytest.mark.gpu
@pytest.mark.parametrize("zw", [0, 93], ids=["symmetric", "zero_point"])
@pytest.mark.parametrize("in_u8", [False, True], ids=["s8", "u8"])
@pytest.mark.parametrize("name,kw", LAYERS, ids=[l[0] for l in LAYERS])
def test_tiles_give_the_plain_kernels_bytes(name, kw, in_u8, zw):
    seed = 97000 + 13 * [l[0] for l in LAYERS].index(name) + 2 * zw + in_u8
    wq = dict(w_dtype=U8, w_offset=zw, per_axis=False) if zw else {}
    c = cases.make_conv_case(name, seed, in_dtype=U8 if in_u8 else S8, in_offset=121 if in_u8 else -7, out_offset=100 if in_u8 else -20, act=cases.RELU6, **wq, **kw)
    kwargs = dict(activation=c.act[0], act_a=c.act[1], act_b=c.act[2], **c.params)
    want = shim.conv2d(c.x, c.w, c.b, c.out_info, algo=shim.ALGO_DIRECT, **kwargs).data
    for tile in range(5000, 5009):
        shim.set_option("igemm_tile", tile)
        try:
            print(name, tile, flush=True)
            got = shim.conv2d(c.x, c.w, c.b, c.out_info, **kwargs)
            kernel = shim.last_kernel()
        finally:
            shim.set_option("igemm_tile", 0)
        print(kernel, flush=True)
        assert kernel.startswith("TapPanelKernel<"), kernel
        np.testing.assert_array_equal(got.data, want, err_msg=f"{tile} {kernel}")


@pytest.mark.gpu
@pytest.mark.parametrize("n,h,ci,co,k,stride,alone,shared", [
    (16, 14, 256, 256, 3, 1, "2, 32, 64, false, false, true", "2, 64, 64, false, false, true"), (9, 28, 72, 96, 3, 1, "2, 32, 64, false, true, false", "2, 64, 64, false, true, false"),
    (16, 28, 128, 128, 3, 1, "2, 64, 128, false, false, true", "2, 64, 64, false, false, true"), (24, 33, 152, 64, 3, 1, "2, 64, 64, false, true, false", "2, 64, 64, false, true, false"),
    (40, 28, 64, 200, 5, 2, "2, 64, 128, false, false, true", "1, 64, 64, false, false, true"), (16, 56, 64, 64, 3, 1, None, "1, 128, 64, false, false, true"),
    (16, 7, 512, 512, 3, 1, "4, 32, 64, false, false, true", "4, 32, 64, false, false, true"), (20, 9, 384, 48, 5, 1, "4, 32, 32, false, false, true", "4, 32, 32, false, false, true"),
    (300, 1, 1024, 1001, 1, 1, "4, 32, 64, false, false, true", "4, 32, 64, false, false, true"), (120, 1, 1040, 3001, 1, 1, "4, 32, 64, false, false, false", "4, 32, 64, false, false, false"),
    (612, 1, 1232, 432, 1, 1, None, None), (1690, 1, 1088, 144, 1, 1, None, None), (85, 1, 1488, 3004, 1, 1, "4, 32, 64, false, false, false", "4, 32, 64, false, false, false"),
    (755, 1, 1848, 397, 1, 1, "4, 32, 64, false, true, false", "4, 32, 64, false, true, false"),
    (1, 28, 128, 512, 1, 1, "2, 32, 64, false, false, true", "2, 32, 64, false, false, true"), (1, 56, 96, 130, 1, 1, "2, 32, 64, false, false, false", "2, 32, 64, false, false, false")])
def test_launches_that_choose_a_tile(n, h, ci, co, k, stride, alone, shared):
    """The automatic choice, with and without launches beside it, on first use inside a captured graph as well."""
    c = cases.make_conv_case("auto", 98000 + ci, n=n, h=h, w=h, ci=ci, co=co, kh=k, kw=k, stride=(stride, stride), act=cases.RELU)
    kwargs = dict(activation=c.act[0], act_a=c.act[1], act_b=c.act[2], **c.params)
    want = shim.conv2d(c.x, c.w, c.b, c.out_info, algo=shim.ALGO_DIRECT, **kwargs).data
    dev = shim.Device()
    x, y, blank = shim.DeviceBuffer(c.x.data.nbytes).upload(c.x.data), shim.DeviceBuffer(want.nbytes), np.zeros_like(want)
    for lanes in (1, 2):
        plan = shim.Conv2dPlan(c.x.info, c.w, c.b, c.out_info, **kwargs)
        plan.set_concurrency(lanes)
        stream = dev.stream()
        dev.graph_begin(stream)
        plan.run(n, x.ptr, y.ptr, stream)
        graph = dev.graph_end(stream)
        kernel, tile = shim.last_kernel(), alone if lanes == 1 else shared
        print(lanes, kernel, flush=True)
        assert kernel == f"TapPanelKernel<{tile}>" if tile else not kernel.startswith("TapPanelKernel<"), kernel
        for _ in range(3):
            y.upload(blank)
            dev.graph_launch(graph, stream)
            dev.stream_sync(stream)
            np.testing.assert_array_equal(y.download(want.shape, want.dtype), want)
        dev.graph_destroy(graph)
        dev.stream_destroy(stream)


@pytest.mark.gpu
@pytest.mark.parametrize("n,h,ci,co,kh,kw,dilation,kernel", [
    (2, 160, 64, 64, 9, 1, 1, "IgemmKernel<128, 64, "), (2, 148, 64, 32, 3, 3, 6, "IgemmKernel<64, 64, "), (1, 224, 256, 64, 3, 3, 1, "IgemmLdsKernel<64, 64, "),
    (2, 56, 64, 64, 32, 1, 1, "SmallConvKernel<"), (2, 56, 256, 64, 3, 3, 4, "SmallConvKernel<"), (1, 24, 448, 288, 2, 2, 1, "SmallConvKernel<"),
    (4, 18, 64, 48, 5, 5, 3, "SmallConvKernel<"), (8, 36, 128, 16, 4, 4, 2, "TapPanelKernel<"), (5, 26, 128, 100, 4, 7, 3, "TapPanelKernel<"),
    (2, 93, 192, 32, 3, 3, 1, "TapPanelKernel<"), (2, 56, 256, 64, 3, 3, 2, "TapPanelKernel<")])
def test_launches_whose_runs_are_long_for_their_outputs(n, h, ci, co, kh, kw, dilation, kernel):
    """They leave the panel to kernels that read pixels per tap, unless those take longer all the same."""
    c = cases.make_conv_case("long", 98500 + ci, n=n, h=h, w=h, ci=ci, co=co, kh=kh, kw=kw, dilation=(dilation, dilation), act=cases.RELU)
    kwargs = dict(activation=c.act[0], act_a=c.act[1], act_b=c.act[2], **c.params)
    got = shim.conv2d(c.x, c.w, c.b, c.out_info, **kwargs)
    print(shim.last_kernel(), flush=True)
    assert shim.last_kernel().startswith(kernel), shim.last_kernel()
    np.testing.assert_array_equal(got.data, shim.conv2d(c.x, c.w, c.b, c.out_info, algo=shim.ALGO_DIRECT, **kwargs).data)


@pytest.mark.gpu
@pytest.mark.parametrize("n,ci,co,kernel", [(16, 128, 48, "TapPanelKernel<"), (2, 128, 48, "TapPanelKernel<"), (40, 80, 48, "TapPanelKernel<"), (16, 128, 40, "Add")])
def test_an_addition_behind(n, ci, co, kernel):
    c = cases.make_conv_case("add", 99000 + ci + n, n=n, h=14, w=14, ci=ci, co=co, in_scale=0.0235, out_scale=0.1, out_offset=3)
    info = TensorInfo(c.out_info.shape, S8, (0.1,), -128)
    other = QTensor(info, synth.uniform_int(52, info.shape, -128, 127, np.int64))
    plan = shim.Conv2dPlan(c.x.info, c.w, c.b, c.out_info, **c.params)
    xd, od = shim.DeviceBuffer(c.x.data.nbytes).upload(c.x.data), shim.DeviceBuffer(other.data.nbytes).upload(other.data)
    mid, both = shim.DeviceBuffer(other.data.nbytes), shim.DeviceBuffer(other.data.nbytes)
    plan.run(n, xd.ptr, mid.ptr)
    assert shim.last_kernel().startswith("TapPanelKernel<"), shim.last_kernel()
    want = shim.add(QTensor(c.out_info, mid.download(info.shape, numpy_dtype(S8))), other, info, activation=shim.ACT_RELU)
    plan.run_add(n, xd.ptr, od.ptr, info, info, both.ptr, activation=shim.ACT_RELU)
    assert shim.last_kernel().startswith(kernel), shim.last_kernel()      # "Add": channels that are no whole pieces leave it a launch of its own
    shim.Device().synchronize()
    np.testing.assert_array_equal(both.download(info.shape, numpy_dtype(S8)), want.data)


@pytest.mark.gpu
@pytest.mark.parametrize("ci,co,k,zw,text", [(64, 64, 3, 0, "; weights in registers or input pixels in LDS where faster"), (64, 65, 3, 0, "; input pixels in LDS for all taps where faster"),
                                             (128, 64, 3, 0, "; input pixels in LDS for all taps where faster"), (128, 64, 3, 93, ", weight zero point by row sums"), (64, 64, 2, 0, "; from 192 row tiles on input tile in LDS for all taps"),
                                             (16, 64, 3, 0, ""), (256, 64, 1, 0, "")])
def test_what_a_plan_says_of_its_launches(ci, co, k, zw, text):
    wq = dict(w_dtype=U8, w_offset=zw, per_axis=False) if zw else {}
    c = cases.make_conv_case("info", 99600 + ci, n=1, h=8, w=8, ci=ci, co=co, kh=k, kw=k, **wq)
    info = shim.Conv2dPlan(c.x.info, c.w, c.b, c.out_info, **c.params).algo()[1]
    assert len(info) < 127 and info.endswith(text) and (text or "in LDS" not in info), info


@pytest.mark.gpu
def test_a_plans_choice_follows_batch_and_lanes():
    """What a plan keeps of its last choice is for that batch and those lanes alone."""
    c = cases.make_conv_case("kept", 99500, n=64, h=14, w=14, ci=64, co=256, act=cases.RELU)
    kwargs = dict(activation=c.act[0], act_a=c.act[1], act_b=c.act[2], **c.params)
    want = shim.conv2d(c.x, c.w, c.b, c.out_info, algo=shim.ALGO_DIRECT, **kwargs).data
    x, y = shim.DeviceBuffer(c.x.data.nbytes).upload(c.x.data), shim.DeviceBuffer(want.nbytes)
    dev = shim.Device()

    def run(plan, n, lanes):
        plan.set_concurrency(lanes)
        y.upload(np.zeros_like(want))
        plan.run(n, x.ptr, y.ptr)
        kernel = shim.last_kernel()
        dev.synchronize()
        np.testing.assert_array_equal(y.download(want.shape, want.dtype)[:n], want[:n], err_msg=f"{n} {lanes} {kernel}")
        return kernel

    calls = [(n, lanes) for n in (64, 1, 16, 7) for lanes in (1, 2)]
    fresh = {call: run(shim.Conv2dPlan(c.x.info, c.w, c.b, c.out_info, **kwargs), *call) for call in calls}
    print(fresh, flush=True)
    assert len(set(fresh.values())) >= 4 and fresh[64, 1].startswith("HeldConvKernel<") and fresh[64, 2].startswith("TapPanelKernel<")
    plan = shim.Conv2dPlan(c.x.info, c.w, c.b, c.out_info, **kwargs)
    for call in calls + calls[::-1] + calls[::3] + calls[:1] * 2:
        assert run(plan, *call) == fresh[call], call
