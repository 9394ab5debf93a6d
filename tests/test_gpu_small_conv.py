"""Layers with few output rows (32 x 32 tiles whose waves split K) against the plain kernel, bit for bit, and the CPU checker:
edges of the tile in rows and channels, K of less than one step up to many, filters, strides, padding, both activation types,
weights with a zero point, channel counts that are no multiple of 16, an Addition behind the layer."""
import numpy as np
import pytest

from armnn_amd import shim, synth
from armnn_amd.tensor import QTensor, TensorInfo, numpy_dtype
from tests import cases
from tests.helpers import lsb_diff

pytestmark = pytest.mark.gpu
U8, S8 = cases.U8, cases.S8

LAYERS = [
    ("one_pixel_k16", dict(n=1, h=1, w=1, ci=16, co=16, kh=1, kw=1)),
    ("five_rows_k48", dict(n=5, h=1, w=1, ci=48, co=33, kh=1, kw=1)),
    ("31_rows_co31", dict(n=1, h=1, w=31, ci=160, co=31, kh=1, kw=1)),
    ("33_rows_co48", dict(n=3, h=11, w=1, ci=208, co=48, kh=1, kw=1)),
    ("7x7_c512_3x3", dict(n=1, h=7, w=7, ci=512, co=512)),
    ("14x14_c256_3x3_s2", dict(n=2, h=14, w=14, ci=256, co=256, stride=(2, 2))),
    ("13x9_c80_5x5_dilated", dict(n=1, h=13, w=9, ci=80, co=96, kh=5, kw=5, dilation=(2, 1))),
    ("7x7_c2048_1x1", dict(n=3, h=7, w=7, ci=2048, co=512, kh=1, kw=1)),
    ("28x28_c128_1x1_slab_plan", dict(n=1, h=28, w=28, ci=128, co=256, kh=1, kw=1)),
    ("14x14_c24_3x3_ragged", dict(n=1, h=14, w=14, ci=24, co=72)),
    ("9x9_c40_1x1_ragged_to_the_end", dict(n=2, h=9, w=9, ci=40, co=17, kh=1, kw=1)),
    ("valid_c7_3x3_ragged", dict(n=1, h=6, w=6, ci=7, co=5, padding="valid")),
]


@pytest.mark.parametrize("zw", [0, 93], ids=["symmetric", "zero_point"])
@pytest.mark.parametrize("in_u8", [False, True], ids=["s8", "u8"])
@pytest.mark.parametrize("name,kw", LAYERS, ids=[l[0] for l in LAYERS])
def test_few_rows(port, name, kw, in_u8, zw):
    seed = 51000 + 13 * [l[0] for l in LAYERS].index(name) + 2 * zw + in_u8
    wq = dict(w_dtype=U8, w_offset=zw, per_axis=False) if zw else {}
    c = cases.make_conv_case(name, seed, in_dtype=U8 if in_u8 else S8, in_offset=121 if in_u8 else -7, out_offset=100 if in_u8 else -20,
                             act=cases.RELU6, **wq, **kw)
    kwargs = dict(activation=c.act[0], act_a=c.act[1], act_b=c.act[2], **c.params)
    got = shim.conv2d(c.x, c.w, c.b, c.out_info, **kwargs)
    kernel = shim.last_kernel()
    print(f"{name}: {kernel}", flush=True)
    panel = "7x7_c512_3x3" == name                       # many whole k-steps: the form with a panel
    assert kernel.startswith("TapPanelKernel<" if panel else "SmallConvKernel<") or c.out_info.num_elements // c.out_info.shape[-1] <= 4, kernel
    np.testing.assert_array_equal(got.data, shim.conv2d(c.x, c.w, c.b, c.out_info, algo=shim.ALGO_DIRECT, **kwargs).data)
    want = port.activation(port.conv2d(c.x, c.w, c.b, c.out_info, **c.params), c.out_info, *c.act)
    mx, exact = lsb_diff(got.data, want.data)
    assert mx <= 1 and exact >= 0.99, (mx, exact)


@pytest.mark.parametrize("n,h,ci,co,k,expected", [(1, 14, 256, 1024, 1, "SmallConvKernel<"), (1, 7, 512, 2048, 1, "SmallConvKernel<"), (1, 9, 128, 48, 2, "SmallConvKernel<"),
                                                  (1, 9, 64, 48, 3, "Add"), (1, 9, 128, 48, 3, "TapPanelKernel<")])
def test_few_rows_with_an_addition_behind(n, h, ci, co, k, expected):
    c = cases.make_conv_case("add", 52000 + co + k, n=n, h=h, w=h, ci=ci, co=co, kh=k, kw=k, in_scale=0.0235, out_scale=0.1, out_offset=3)
    info = TensorInfo(c.out_info.shape, S8, (0.1,), -128)
    other = QTensor(info, synth.uniform_int(52, info.shape, -128, 127, np.int64))
    dev = shim.Device()
    plan = shim.Conv2dPlan(c.x.info, c.w, c.b, c.out_info, **c.params)
    xd, od = shim.DeviceBuffer(c.x.data.nbytes).upload(c.x.data), shim.DeviceBuffer(other.data.nbytes).upload(other.data)
    mid, both = shim.DeviceBuffer(other.data.nbytes), shim.DeviceBuffer(other.data.nbytes)
    plan.run(n, xd.ptr, mid.ptr)
    want = shim.add(QTensor(c.out_info, mid.download(info.shape, numpy_dtype(S8))), other, info, activation=shim.ACT_RELU)
    plan.run_add(n, xd.ptr, od.ptr, info, info, both.ptr, activation=shim.ACT_RELU)
    kernel = shim.last_kernel()
    dev.synchronize()
    assert kernel.startswith(expected), kernel
    np.testing.assert_array_equal(both.download(info.shape, numpy_dtype(S8)), want.data)


@pytest.mark.parametrize("zw", [0, 93], ids=["symmetric", "zero_point"])
@pytest.mark.parametrize("ci,k,stride,walk", [
    (16, 5, 1, "false, false"), (48, 3, 1, "false, false"), (64, 3, 1, "false, true"), (112, 5, 1, "false, false"), (192, 3, 2, "false, true"), (272, 5, 1, "false, false"),
    (64, 4, 1, "false, false"), (128, 5, 2, "false, false"), (320, 1, 1, "false, true"), (24, 5, 1, "true, false"), (72, 3, 1, "true, false"), (250, 5, 1, "true, false"),
    (192, 3, 1, None), (320, 5, 1, None)])
def test_walks_over_the_taps(ci, k, stride, walk, zw):
    """Taps of whole steps of 64 bytes, of other multiples of 16 and of any size, shorter and longer than a step, each wave's start inside
    a tap or at one's end.  Many whole k-steps at stride 1 take the form with a panel."""
    wq = dict(w_dtype=U8, w_offset=zw, per_axis=False) if zw else {}
    c = cases.make_conv_case("walk", 53000 + ci + zw, n=2, h=9, w=7, ci=ci, co=36, kh=k, kw=k, stride=(stride, stride), out_offset=-20, act=cases.RELU6, **wq)
    kwargs = dict(activation=c.act[0], act_a=c.act[1], act_b=c.act[2], **c.params)
    got = shim.conv2d(c.x, c.w, c.b, c.out_info, **kwargs)
    kernel = shim.last_kernel()
    print(ci, k, kernel, flush=True)
    aw = "true" if zw else "false"
    assert kernel == (f"SmallConvKernel<{aw}, {walk}>" if walk else f"TapPanelKernel<4, 32, 32, {aw}, false, true>")
    np.testing.assert_array_equal(got.data, shim.conv2d(c.x, c.w, c.b, c.out_info, algo=shim.ALGO_DIRECT, **kwargs).data)
