"""Convolutions whose waves hold the weights of nine taps over 64 channels in registers (csrc/held_conv_kernel.h), at the edges of their groups of 16
pixels, of their tiles of 64 channels and of both lengths of a block's run, against the plain kernel, bit for bit."""
import numpy as np
import pytest

from armnn_amd import shim
from tests import cases

U8, S8 = cases.U8, cases.S8

LAYERS = [
    ("one_pixel", dict(n=1, h=1, w=1, co=16)),
    ("65_pixels_two_columns", dict(n=5, h=1, w=13, co=144)),
    ("images_of_9_pixels", dict(n=15, h=3, w=3, co=64)),
    ("valid", dict(n=1, h=7, w=47, co=80, padding="valid")),
    ("stride_2", dict(n=3, h=15, w=9, co=48, stride=(2, 2))),
    ("dilated", dict(n=2, h=13, w=9, co=32, dilation=(2, 1))),
    ("padding_at_two_sides", dict(n=2, h=6, w=7, co=64, padding=(2, 0, 1, 0))),
    ("filter_1x9", dict(n=2, h=5, w=30, co=64, kh=1, kw=9)),
    ("first_row_in_the_padding", dict(n=1, h=9, w=200, co=64, kh=1, kw=9, stride=(2, 2), padding=(1, 0, 4, 4))),
    ("wide_rows", dict(n=1, h=5, w=224, co=64)),                       # the longer run
    ("more_blocks_than_fit", dict(n=100, h=23, w=23, co=528)),
]


@pytest.mark.gpu
@pytest.mark.parametrize("in_u8", [False, True], ids=["s8", "u8"])
@pytest.mark.parametrize("name,kw", LAYERS, ids=[l[0] for l in LAYERS])
def test_weights_in_registers_give_the_plain_kernels_bytes(name, kw, in_u8):
    c = cases.make_conv_case(name, 96000 + 2 * [l[0] for l in LAYERS].index(name) + in_u8, ci=64, in_dtype=U8 if in_u8 else S8, in_offset=121 if in_u8 else -7,
                             out_offset=100 if in_u8 else -20, act=cases.RELU6, **kw)
    kwargs = dict(activation=c.act[0], act_a=c.act[1], act_b=c.act[2], **c.params)
    want = shim.conv2d(c.x, c.w, c.b, c.out_info, algo=shim.ALGO_DIRECT, **kwargs).data
    shim.set_option("igemm_tile", 5009)
    try:
        got = shim.conv2d(c.x, c.w, c.b, c.out_info, **kwargs)
    finally:
        shim.set_option("igemm_tile", 0)
    kernel = shim.last_kernel()
    print(name, kernel, flush=True)
    assert kernel.startswith("HeldConvKernel<"), kernel
    np.testing.assert_array_equal(got.data, want)


@pytest.mark.gpu
@pytest.mark.parametrize("n,h,co,taken", [(6, 56, 64, "4"), (32, 56, 64, "10"), (40, 28, 192, "4"), (3, 56, 64, None), (1, 112, 128, None), (6, 56, 65, None),
                                             (1, 208, 64, "10"), (3, 150, 64, "10"), (3, 208, 64, "10"), (1, 224, 256, None), (3, 256, 64, None), (1, 300, 64, None)])
def test_launches_that_choose_it(n, h, co, taken):
    """... but not where rows are so wide that several rounds of blocks would each fetch a long run for few outputs."""
    c = cases.make_conv_case("auto", 96100 + n, n=n, h=h, w=h, ci=64, co=co, act=cases.RELU)
    kwargs = dict(activation=c.act[0], act_a=c.act[1], act_b=c.act[2], **c.params)
    want = shim.conv2d(c.x, c.w, c.b, c.out_info, algo=shim.ALGO_DIRECT, **kwargs).data
    got = shim.conv2d(c.x, c.w, c.b, c.out_info, **kwargs)
    kernel = shim.last_kernel()
    print(kernel, flush=True)
    assert kernel.startswith(f"HeldConvKernel<4, {taken}, ") if taken else not kernel.startswith("HeldConvKernel<"), kernel
    np.testing.assert_array_equal(got.data, want)
