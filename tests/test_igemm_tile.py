"""Tiles of the implicit GEMM (csrc/igemm_tile.h) lie inside the channels that a plan pads to: blocks read weights and constants for all
channels of their tile.  The rule over sizes on the CPU, the shapes that it turns on against the plain kernel on the device."""
import os
import subprocess

import numpy as np
import pytest

from armnn_amd import shim
from tests import cases
from tests.conftest import ROOT

PROGRAM = r"""
#include "igemm_tile.h"
#include <initializer_list>
#include <cstdio>
int main()
{
    int bad = 0;
    for (int forced : {0, 64, 96, 128, 256, 512})
        for (int narrow = 0; narrow < 2; ++narrow)
            for (long long pixels : {1ll, 49ll, 6400ll, 24576ll, 25000ll, 100352ll, 802816ll})
                for (int channels = 1; channels <= 2100; ++channels)
                {
                    const int padded = (channels + 127) / 128 * 128, tile = mi355x::IgemmTile(forced, narrow != 0, pixels, channels, padded);
                    const int width = tile <= 96 ? 64 : tile <= 256 ? 128 : 256;
                    if ((channels + width - 1) / width * width > padded && ++bad < 5)
                        std::printf("%lld pixels, %d channels, forced %d: tile %d past %d channels\n", pixels, channels, forced, tile, padded);
                    if (padded % 256 == 0 && forced == 512 && tile != 512) ++bad;
                }
    return bad != 0;
}
"""


def test_tiles_end_inside_the_padded_channels(tmp_path):
    src, exe = tmp_path / "tile.cpp", tmp_path / "tile"
    src.write_text(PROGRAM)
    subprocess.run(["g++", "-O2", "-std=c++17", "-Wall", "-Werror", f"-I{os.path.join(ROOT, 'armnn_amd', 'csrc')}", str(src), "-o", str(exe)], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout


@pytest.mark.gpu
@pytest.mark.parametrize("co,tile,name", [(300, 0, "IgemmLdsKernel<128, 128"), (300, 512, "IgemmLdsKernel<128, 128"), (500, 512, "IgemmLdsKernel<256, 256")])
def test_filters_of_many_taps(co, tile, name):
    c = cases.make_conv_case("taps49", 96000 + co, n=2, h=112, w=112, ci=128, co=co, kh=7, kw=7, act=cases.RELU6)
    kwargs = dict(activation=c.act[0], act_a=c.act[1], act_b=c.act[2], **c.params)
    shim.set_option("igemm_tile", tile)
    try:
        got = shim.conv2d(c.x, c.w, c.b, c.out_info, **kwargs)
        kernel = shim.last_kernel()
    finally:
        shim.set_option("igemm_tile", 0)
    print(co, tile, kernel, flush=True)
    assert kernel.startswith(name), kernel
    np.testing.assert_array_equal(got.data, shim.conv2d(c.x, c.w, c.b, c.out_info, algo=shim.ALGO_DIRECT, **kwargs).data)
