"""Channel counts that are no multiple of 16, through AUTO against the plain kernel (bit for bit) and the CPU checker.

Sizes are where a padded filter tap or a ragged output row can go wrong: the last pixels of the tensor (their 16-byte chunks
would end beyond it), tensors of little more than 16 bytes, taps that straddle k-tiles, one channel above and below a
multiple of 16, output rows of every length modulo 16, launches for each tile size."""
import numpy as np
import pytest

from armnn_amd import shim
from tests import cases
from tests.helpers import lsb_diff

pytestmark = pytest.mark.gpu
U8, S8 = cases.U8, cases.S8

CONVS = [
    ("1x1_c24_48", dict(n=3, h=11, w=13, ci=24, co=48, kh=1, kw=1)),
    ("1x1_c8_17", dict(n=1, h=1, w=2, ci=8, co=17, kh=1, kw=1)),
    ("1x1_c5_one_image_of_20_bytes", dict(n=2, h=2, w=2, ci=5, co=3, kh=1, kw=1)),
    ("1x1_c17_15", dict(n=4, h=6, w=7, ci=17, co=15, kh=1, kw=1)),
    ("1x1_c200_255", dict(n=2, h=13, w=13, ci=200, co=255, kh=1, kw=1)),
    ("1x1_s2_c40_80", dict(n=2, h=9, w=9, ci=40, co=80, kh=1, kw=1, stride=(2, 2))),
    ("3x3_s2_c72_120", dict(n=2, h=19, w=19, ci=72, co=120, stride=(2, 2))),
    ("3x3_c31_33", dict(n=1, h=10, w=9, ci=31, co=33)),
    ("3x3_c33_31_dilated", dict(n=1, h=15, w=12, ci=33, co=31, dilation=(2, 2))),
    ("3x3_valid_c6_64", dict(n=2, h=8, w=8, ci=6, co=64, padding="valid")),
    ("5x5_c20_24_asymmetric", dict(n=1, h=12, w=15, ci=20, co=24, kh=5, kw=5, padding=(1, 3, 0, 4))),
    ("3x3_c104_136_tiles_of_128", dict(n=8, h=57, w=55, ci=104, co=136)),
    ("3x3_c12_40_tiles_of_128x64", dict(n=12, h=64, w=64, ci=12, co=40)),
    # whole chunks of input, ragged rows of output, on the other kernels
    ("1x1_c64_66", dict(n=2, h=20, w=20, ci=64, co=66, kh=1, kw=1)),
    ("1x1_c256_1001", dict(n=2, h=9, w=9, ci=256, co=1001, kh=1, kw=1)),
    ("3x3_c64_57_resident_tile", dict(n=8, h=56, w=56, ci=64, co=57)),
    ("3x3_c128_79_large_tile", dict(n=8, h=90, w=90, ci=128, co=79)),
    ("3x3_c256_99_k_split", dict(n=1, h=14, w=14, ci=256, co=99)),
]


@pytest.mark.parametrize("in_u8", [False, True], ids=["s8", "u8"])
@pytest.mark.parametrize("zw", [0, 93], ids=["symmetric", "zero_point"])
@pytest.mark.parametrize("name,kw", CONVS, ids=[c[0] for c in CONVS])
def test_ragged_convolutions(port, name, kw, zw, in_u8):
    seed = 41000 + 11 * [c[0] for c in CONVS].index(name) + 2 * zw + in_u8
    wq = dict(w_dtype=U8, w_offset=zw, per_axis=False) if zw else {}
    c = cases.make_conv_case(name, seed, in_dtype=U8 if in_u8 else S8, in_offset=121 if in_u8 else -7, out_offset=100 if in_u8 else -20,
                             act=cases.RELU6, **wq, **kw)
    kwargs = dict(activation=c.act[0], act_a=c.act[1], act_b=c.act[2], **c.params)
    got = shim.conv2d(c.x, c.w, c.b, c.out_info, **kwargs)
    print(f"{name}: {shim.last_kernel()}", flush=True)
    np.testing.assert_array_equal(got.data, shim.conv2d(c.x, c.w, c.b, c.out_info, algo=shim.ALGO_DIRECT, **kwargs).data)
    if got.data.size <= 200000:
        want = port.activation(port.conv2d(c.x, c.w, c.b, c.out_info, **c.params), c.out_info, *c.act)
        mx, exact = lsb_diff(got.data, want.data)
        assert mx <= 1 and exact >= 0.99, (mx, exact)


@pytest.mark.parametrize("m,k,o", [(1, 17, 5), (4, 100, 33), (5, 1000, 10), (64, 999, 1001), (65, 130, 127), (300, 72, 91), (2000, 520, 260)])
@pytest.mark.parametrize("zw", [0, 93], ids=["symmetric", "zero_point"])
def test_ragged_fully_connected(port, m, k, o, zw):
    wq = dict(w_dtype=U8, w_offset=zw, per_axis=False) if zw else {}
    f = cases.make_fc_case("fc", 42000 + m + k + o, m=m, k=k, o=o, in_dtype=U8, in_offset=63, out_offset=30, **wq)
    got = shim.fully_connected(f.x, f.w, f.b, f.out_info)
    print(f"{m}x{k}x{o}: {shim.last_kernel()}", flush=True)
    np.testing.assert_array_equal(got.data, shim.fully_connected(f.x, f.w, f.b, f.out_info, algo=shim.ALGO_DIRECT).data)
    mx, exact = lsb_diff(got.data, port.fully_connected(f.x, f.w, f.b, f.out_info).data)
    assert mx <= 1 and exact >= 0.99, (mx, exact)


def test_tensors_at_any_address():
    """A layer whose channel counts are no multiples of 16 takes tensors at any byte, as the plain kernel always did."""
    import ctypes as C
    c = cases.make_conv_case("any_address", 43000, n=2, h=9, w=7, ci=24, co=32, act=cases.RELU)
    plan = shim.Conv2dPlan(c.x.info, c.w, c.b, c.out_info, activation=c.act[0], act_a=c.act[1], act_b=c.act[2], **c.params)
    want = shim.conv2d(c.x, c.w, c.b, c.out_info, activation=c.act[0], act_a=c.act[1], act_b=c.act[2], algo=shim.ALGO_DIRECT, **c.params)
    for shift in (0, 1, 3, 6, 13):
        xd, yd = shim.DeviceBuffer(c.x.data.nbytes + shift), shim.DeviceBuffer(want.data.nbytes + shift)
        shim._chk(xd.lib.mi355x_memcpy_h2d(xd.ptr + shift, c.x.data.ctypes.data, c.x.data.nbytes, None))
        plan.run(2, xd.ptr + shift, yd.ptr + shift)
        out = np.empty_like(want.data)
        shim._chk(xd.lib.mi355x_memcpy_d2h(out.ctypes.data_as(C.c_void_p), yd.ptr + shift, out.nbytes, None))
        np.testing.assert_array_equal(out, want.data, err_msg=f"shift {shift}")
