"""Three-channel stems at stride 2 through AUTO against the plain kernel, bit for bit.

Sizes are where the kernel's twelve-byte loads and its tiles can go wrong: images whose first and last pixels end the tensor, fewer pixels
than a load or a tile, tiles of 8 and of 16 rows, every width modulo 4, filters narrower and wider than their operand rows allow, output channels around 32 and
64, two halves of the weights."""
import numpy as np
import pytest

from armnn_amd import shim
from tests import cases

pytestmark = pytest.mark.gpu
U8, S8 = cases.U8, cases.S8

STEMS = [
    ("3x3_same_32", dict(n=3, h=37, w=45, co=32, kh=3, kw=3), True),
    ("3x3_same_24_dwords", dict(n=2, h=33, w=34, co=24, kh=3, kw=3), True),
    ("3x3_valid_64", dict(n=2, h=19, w=67, co=64, kh=3, kw=3, padding="valid"), True),
    ("3x3_valid_36", dict(n=1, h=3, w=3, co=36, kh=3, kw=3, padding="valid"), True),
    ("3x4_asymmetric", dict(n=2, h=18, w=70, co=40, kh=3, kw=4, padding=(0, 2, 3, 1)), True),
    ("3x1", dict(n=1, h=21, w=131, co=32, kh=3, kw=1), True),
    ("3x3_one_pixel", dict(n=1, h=1, w=1, co=16, kh=3, kw=3), False),
    ("3x3_twelve_bytes", dict(n=1, h=2, w=2, co=16, kh=3, kw=3), True),
    ("3x3_four_images_of_a_pixel", dict(n=4, h=1, w=1, co=16, kh=3, kw=3), True),
    ("7x7_same_64", dict(n=2, h=45, w=50, co=64, kh=7, kw=7), True),
    ("7x7_padding_3_32", dict(n=2, h=31, w=63, co=32, kh=7, kw=7, padding=(3, 3, 3, 3)), True),
    ("7x7_valid_60", dict(n=1, h=9, w=35, co=60, kh=7, kw=7, padding="valid"), True),
    ("7x8", dict(n=1, h=17, w=33, co=64, kh=7, kw=8), True),
    ("7x5_wide_padding", dict(n=2, h=8, w=5, co=48, kh=7, kw=5, padding=(6, 5, 4, 4)), True),
    ("7x7_tiles_of_16_rows", dict(n=40, h=130, w=200, co=64, kh=7, kw=7), True),     # (768 tiles of 16 rows or more; the last has one)
    ("7x7_tiles_of_16_rows_32", dict(n=40, h=130, w=200, co=32, kh=7, kw=7), True),
    ("3x3_tiles_of_16_rows", dict(n=32, h=130, w=260, co=32, kh=3, kw=3), True),
    ("3x3_tiles_of_16_rows_64", dict(n=32, h=130, w=260, co=64, kh=3, kw=3), True),
]


@pytest.mark.parametrize("in_u8", [False, True], ids=["s8", "u8"])
@pytest.mark.parametrize("weights", ["per_axis", "two_halves"])
@pytest.mark.parametrize("name,kw,taken", STEMS, ids=[s[0] for s in STEMS])
def test_rgb_stems(name, kw, taken, weights, in_u8):
    wq = dict(per_axis=False, w_dtype=U8, w_offset=151, w_std=70.0) if weights == "two_halves" else {}
    seed = 52000 + 7 * [s[0] for s in STEMS].index(name) + in_u8
    c = cases.make_conv_case(name, seed, ci=3, stride=(2, 2), in_dtype=U8 if in_u8 else S8, in_offset=131 if in_u8 else -9, in_scale=0.02, out_scale=0.1,
                             out_offset=7, act=cases.RELU6 if kw["co"] % 8 else (0, 0.0, 0.0), **wq, **kw)
    kwargs = dict(activation=c.act[0], act_a=c.act[1], act_b=c.act[2], **c.params)
    got = shim.conv2d(c.x, c.w, c.b, c.out_info, **kwargs)
    kernel = shim.last_kernel()
    print(f"{name}: {kernel}", flush=True)
    assert kernel.startswith("StemRgbKernel") == (taken and (weights == "per_axis" or kw["kh"] == 3))
    if kernel.startswith("StemRgbKernel"):
        halves = weights == "two_halves"                  # always in tiles of 16 rows
        rows = 16 if halves or "16_rows" in name else 8
        assert kernel == f"StemRgbKernel<{kw['kh']}, {1 if kw['co'] <= 32 else 2}, {rows}, {'true' if halves else 'false'}>"
    np.testing.assert_array_equal(got.data, shim.conv2d(c.x, c.w, c.b, c.out_info, algo=shim.ALGO_DIRECT, **kwargs).data)
