"""1x1 convolutions of many rows (whole rows in LDS, weights in operand order) against the plain kernel, bit for bit: rows and
channels that are no whole tiles, K of less than one step up to more than one panel, both activation types, weights with a zero
point, an Addition behind the layer."""
import numpy as np
import pytest

from armnn_amd import shim, synth
from armnn_amd.tensor import QTensor, TensorInfo, numpy_dtype
from tests import cases

pytestmark = pytest.mark.gpu
U8, S8 = cases.U8, cases.S8

# rows (n, h, w), input channels, output channels, instance
LAYERS = [
    (1, 121, 121, 16, 48, "1, 128"),
    (4, 64, 65, 64, 64, "1, 128"),
    (1, 110, 113, 112, 144, "2, 128"),
    (9, 29, 31, 128, 256, "2, 128"),
    (3, 80, 79, 144, 32, "1, 256"),
    (5, 41, 43, 256, 208, "2, 256"),
    (1, 1, 12300, 272, 240, "2, 512"),
    (4, 80, 77, 512, 64, "1, 512"),
    (1, 1, 4100, 560, 688, "2, 512"),
    (2, 61, 67, 768, 400, "2, 512"),
]


@pytest.mark.parametrize("addition", [False, True], ids=["alone", "addition"])
@pytest.mark.parametrize("zw", [0, 93], ids=["symmetric", "zero_point"])
@pytest.mark.parametrize("n,h,w,ci,co,instance", LAYERS, ids=[f"{l[0] * l[1] * l[2]}x{l[3]}_{l[4]}" for l in LAYERS])
def test_many_rows(n, h, w, ci, co, instance, zw, addition):
    dt = U8 if (ci // 16 + co // 16) % 2 else S8
    wq = dict(w_dtype=U8, w_offset=zw, per_axis=False) if zw else {}
    c = cases.make_conv_case("rows", 71000 + ci + co + zw, n=n, h=h, w=w, ci=ci, co=co, kh=1, kw=1, in_dtype=dt, in_scale=0.0235,
                             in_offset=121 if dt == U8 else -7, out_scale=0.1, out_offset=100 if dt == U8 else -20, act=cases.RELU6 if not addition else (0, 0.0, 0.0), **wq)
    dev = shim.Device()
    kwargs = dict(activation=c.act[0], act_a=c.act[1], act_b=c.act[2], **c.params)
    plan = shim.Conv2dPlan(c.x.info, c.w, c.b, c.out_info, **kwargs)
    want = shim.conv2d(c.x, c.w, c.b, c.out_info, algo=shim.ALGO_DIRECT, **kwargs)
    xd = shim.DeviceBuffer(c.x.data.nbytes).upload(c.x.data)
    yd = shim.DeviceBuffer(c.out_info.num_elements)
    info = c.out_info
    if addition:
        info = TensorInfo(c.out_info.shape, dt, (0.09,), 90 if dt == U8 else -100)
        other = QTensor(info, synth.uniform_int(53, info.shape, 0 if dt == U8 else -128, 255 if dt == U8 else 127, np.int64))
        want = shim.add(want, other, info, activation=shim.ACT_RELU)
        od = shim.DeviceBuffer(other.data.nbytes).upload(other.data)
        plan.run_add(n, xd.ptr, od.ptr, info, info, yd.ptr, activation=shim.ACT_RELU)
    else:
        plan.run(n, xd.ptr, yd.ptr)
    kernel = shim.last_kernel()
    print(kernel, flush=True)
    assert kernel == f"RowPanelKernel<{instance}, {'true' if zw else 'false'}>", kernel
    dev.synchronize()
    got = yd.download(info.shape, numpy_dtype(dt))
    assert len(np.unique(got)) > 8
    np.testing.assert_array_equal(got, want.data)
