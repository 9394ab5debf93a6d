"""Depthwise 3x3 + pointwise 1x1 in one launch with the layer between in LDS: the bytes of the two layers run apart, over the
kernel's instances, maps that are no whole tiles, channel counts that are no whole blocks, weights with a zero point."""
import numpy as np
import pytest

from armnn_amd import shim
from armnn_amd.tensor import QTensor, numpy_dtype
from tests import cases
from tests.helpers import lsb_diff

pytestmark = pytest.mark.gpu
U8, S8 = cases.U8, cases.S8

# n, h, w, channels, output channels, stride: the tile that the launch's size asks for
PAIRS = [
    (1, 3, 5, 16, 16, 1, "4, 4, 8, 1, 0"),
    (1, 9, 6, 48, 80, 2, "4, 4, 8, 1, 0"),
    (1, 7, 7, 1024, 1024, 1, "4, 4, 8, 1, 0"),
    (4, 14, 14, 512, 512, 1, "4, 4, 16, 1, 0"),
    (13, 27, 30, 192, 208, 2, "4, 8, 8, 2, 0"),
    (8, 20, 22, 192, 192, 1, "4, 8, 8, 2, 0"),
    (5, 28, 28, 256, 256, 1, "4, 8, 8, 2, 4"),
    (7, 14, 14, 512, 512, 1, "4, 8, 8, 2, 8"),
    (14, 28, 27, 256, 512, 2, "4, 8, 8, 4, 4"),
    (14, 14, 14, 512, 512, 1, "4, 8, 8, 4, 8"),
    (27, 14, 13, 512, 1024, 2, "4, 8, 8, 4, 8"),
    (14, 28, 28, 256, 256, 1, "8, 8, 8, 2, 4"),
    (52, 13, 14, 256, 512, 1, "8, 8, 8, 4, 4"),
    (52, 14, 14, 512, 512, 1, "8, 8, 8, 4, 8"),
    (4, 60, 50, 16, 48, 1, "8, 16, 4, 1, 1"),
    (9, 65, 70, 48, 96, 2, "8, 16, 4, 2, 1"),
    (4, 41, 44, 96, 96, 1, "8, 8, 4, 2, 2"),
    (8, 60, 61, 112, 192, 2, "8, 8, 4, 4, 2"),
    (1024, 7, 8, 128, 128, 1, "8, 8, 4, 2, 2"),
    (1024, 13, 15, 128, 256, 2, "8, 8, 4, 4, 2"),
]


@pytest.mark.parametrize("general", [False, True], ids=["symmetric", "zero_points"])
@pytest.mark.parametrize("n,h,w,c,co,s,tile", PAIRS, ids=[f"{p[0]}x{p[1]}x{p[2]}x{p[3]}_{p[4]}_s{p[5]}" for p in PAIRS])
def test_pair_equals_the_layers_run_apart(n, h, w, c, co, s, tile, general):
    dt, mid_zp = (U8, 0) if (c + h) % 2 else (S8, -128)
    wq = dict(w_dtype=U8, w_offset=101, per_axis=False) if general else {}
    dw = cases.make_conv_case("dw", 61000 + c + h, n=n, h=h, w=w, ci=c, depthwise=True, stride=(s, s), in_dtype=dt, in_scale=0.0235,
                              in_offset=120 if dt == U8 else -8, out_scale=0.0235, out_offset=mid_zp, act=cases.RELU6,
                              **(dict(wq, w_scale_range=(0.01, 0.02)) if general else dict(w_scale_range=(0.01, 0.05))))
    ho, wo = dw.out_info.shape[1:3]
    pw = cases.make_conv_case("pw", 62000 + co + h, n=n, h=ho, w=wo, ci=c, co=co, kh=1, kw=1, in_dtype=dt, in_scale=0.0235, in_offset=mid_zp,
                              out_scale=0.03, out_offset=mid_zp + 5, act=cases.RELU6 if h % 2 else (0, 0.0, 0.0), **wq)
    dev = shim.Device()

    def plan(case):
        return shim.Conv2dPlan(case.x.info, case.w, case.b, case.out_info, activation=case.act[0], act_a=case.act[1], act_b=case.act[2], **case.params)
    first, second = plan(dw), plan(pw)
    assert first.fusable_with(second), shim.load_library().mi355x_last_error().decode()
    x = shim.DeviceBuffer(dw.x.data.nbytes).upload(dw.x.data)
    mid = shim.DeviceBuffer(dw.out_info.num_elements)
    apart, one = shim.DeviceBuffer(pw.out_info.num_elements), shim.DeviceBuffer(pw.out_info.num_elements)
    first.run_fused(second, n, x.ptr, one.ptr)
    kernel = shim.last_kernel()
    print(kernel, flush=True)
    assert kernel == f"DwPwPanelKernel<{s}, {tile}, {'true' if general else 'false'}>", kernel
    first.run(n, x.ptr, mid.ptr)
    second.run(n, mid.ptr, apart.ptr)
    dev.synchronize()
    got, want = (b.download(pw.out_info.shape, numpy_dtype(dt)) for b in (one, apart))
    assert len(np.unique(want)) > 8
    np.testing.assert_array_equal(got, want)


# n, h, w, channels, output channels, stride, and the layer between's type, scale, zero point and activation, whose lowest or highest code
# lies inside the type: the last block of 64 channels is no whole one in any of them
CLAMPED = [
    (1, 7, 9, 16, 32, 1, U8, 0.1, 0, cases.RELU6),
    (1, 9, 6, 48, 80, 2, S8, 0.05, 20, cases.RELU),
    (8, 20, 22, 176, 192, 1, U8, 0.05, 140, cases.RELU),
    (5, 28, 28, 208, 256, 1, S8, 0.1, -100, cases.RELU6),
    (14, 14, 14, 464, 512, 1, U8, 0.1, 0, cases.RELU6),
    (4, 60, 50, 32, 48, 1, S8, 0.05, 20, cases.RELU),
    (9, 65, 70, 48, 96, 2, U8, 0.05, 140, cases.RELU),
    (8, 60, 61, 112, 192, 2, S8, 0.05, 20, cases.RELU),
]


@pytest.mark.parametrize("n,h,w,c,co,s,dt,scale,zp,act", CLAMPED, ids=[f"{p[0]}x{p[1]}x{p[2]}x{p[3]}_{p[4]}_s{p[5]}" for p in CLAMPED])
def test_channels_that_do_not_exist_count_for_nothing_under_a_clamp(port, n, h, w, c, co, s, dt, scale, zp, act):
    """Weights with a zero point need the sum of a pixel's codes: those past the last channel must not be in it, whatever code
    the activation between the layers turns them into."""
    wq = dict(w_dtype=U8, w_offset=101, per_axis=False)
    dw = cases.make_conv_case("dw", 63000 + c + h, n=n, h=h, w=w, ci=c, depthwise=True, stride=(s, s), in_dtype=dt, in_scale=0.0235,
                              in_offset=120 if dt == U8 else -8, out_scale=scale, out_offset=zp, act=act, w_scale_range=(0.01, 0.02), **wq)
    ho, wo = dw.out_info.shape[1:3]
    pw = cases.make_conv_case("pw", 64000 + co + h, n=n, h=ho, w=wo, ci=c, co=co, kh=1, kw=1, in_dtype=dt, in_scale=scale, in_offset=zp,
                              out_scale=0.3, out_offset=100 if dt == U8 else -20, **wq)
    dev = shim.Device()

    def plan(case):
        return shim.Conv2dPlan(case.x.info, case.w, case.b, case.out_info, activation=case.act[0], act_a=case.act[1], act_b=case.act[2], **case.params)
    first, second = plan(dw), plan(pw)
    assert first.fusable_with(second), shim.load_library().mi355x_last_error().decode()
    x = shim.DeviceBuffer(dw.x.data.nbytes).upload(dw.x.data)
    mid = shim.DeviceBuffer(dw.out_info.num_elements)
    apart, one = shim.DeviceBuffer(pw.out_info.num_elements), shim.DeviceBuffer(pw.out_info.num_elements)
    first.run_fused(second, n, x.ptr, one.ptr)
    kernel = shim.last_kernel()
    print(kernel, flush=True)
    assert kernel.startswith(f"DwPwPanelKernel<{s}, ") and kernel.endswith("true>"), kernel
    first.run(n, x.ptr, mid.ptr)
    second.run(n, mid.ptr, apart.ptr)
    dev.synchronize()
    got, want = (b.download(pw.out_info.shape, numpy_dtype(dt)) for b in (one, apart))
    assert len(np.unique(want)) > 8
    np.testing.assert_array_equal(got, want)
    if n == 1:
        between = port.activation(port.conv2d(dw.x, dw.w, dw.b, dw.out_info, **dw.params), dw.out_info, *dw.act)
        ref = port.conv2d(QTensor(pw.x.info, between.data), pw.w, pw.b, pw.out_info, **pw.params)
        mx, exact = lsb_diff(got, ref.data)
        assert mx <= 1 and exact >= 0.99, (mx, exact)


def _pair(seed, n, h, c, co, **wq):
    scales = dict(w_scale_range=(0.01, 0.02)) if wq else dict(w_scale_range=(0.01, 0.05))
    dw = cases.make_conv_case("dw", seed, n=n, h=h, w=h, ci=c, depthwise=True, in_dtype=U8, in_scale=0.0235, in_offset=120, out_scale=0.0235,
                              out_offset=0, act=cases.RELU6, **scales, **wq)
    pw = cases.make_conv_case("pw", seed + 9, n=n, h=h, w=h, ci=c, co=co, kh=1, kw=1, in_dtype=U8, in_scale=0.0235, in_offset=0, out_scale=0.03,
                              out_offset=5, **wq)
    plans = [shim.Conv2dPlan(q.x.info, q.w, q.b, q.out_info, activation=q.act[0], act_a=q.act[1], act_b=q.act[2], **q.params) for q in (dw, pw)]
    return dw, pw, plans


@pytest.mark.parametrize("asked", [False, True], ids=["first_run", "after_fusion_pays"])
def test_constants_of_the_pair_are_built_at_first_use_also_under_capture_and_from_two_threads(asked):
    import threading
    dev = shim.Device()
    n, h, c, co = 3, 14, 208, 192
    dw, pw, (first, second) = _pair(65000, n, h, c, co, w_dtype=U8, w_offset=101, per_axis=False)
    streams = [dev.stream(), dev.stream()]
    x = shim.DeviceBuffer(dw.x.data.nbytes).upload(dw.x.data)
    mid, apart = shim.DeviceBuffer(dw.out_info.num_elements), shim.DeviceBuffer(pw.out_info.num_elements)
    first.run(n, x.ptr, mid.ptr)
    second.run(n, mid.ptr, apart.ptr)
    dev.synchronize()
    want = apart.download(pw.out_info.shape, numpy_dtype(U8))
    # captured: the building does not go into the graph
    one = shim.DeviceBuffer(pw.out_info.num_elements)
    if asked:
        assert first.fusion_pays(second, n)
    dev.graph_begin(streams[0])
    first.run_fused(second, n, x.ptr, one.ptr, streams[0])
    assert shim.last_kernel().startswith("DwPwPanelKernel<1, ")
    graph = dev.graph_end(streams[0])
    for fill in (0, 255, 7):
        shim._chk(one.lib.mi355x_fill_u8(one.ptr, fill, pw.out_info.num_elements, streams[0]))
        dev.graph_launch(graph, streams[0])
        np.testing.assert_array_equal(one.download(pw.out_info.shape, numpy_dtype(U8), streams[0]), want)
    dev.graph_destroy(graph)
    # two threads meet at the same fresh plans
    _, _, (first, second) = _pair(65000, n, h, c, co, w_dtype=U8, w_offset=101, per_axis=False)
    outs, errors, start = [shim.DeviceBuffer(pw.out_info.num_elements) for _ in range(2)], [], threading.Barrier(2)

    def work(k):
        try:
            start.wait()
            if asked:
                first.fusion_pays(second, n)
            first.run_fused(second, n, x.ptr, outs[k].ptr, streams[k])
            dev.stream_sync(streams[k])
        except Exception as e:                             # pragma: no cover
            errors.append(e)
    threads = [threading.Thread(target=work, args=(k,)) for k in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not errors, errors
    for o in outs:
        np.testing.assert_array_equal(o.download(pw.out_info.shape, numpy_dtype(U8)), want)


def test_plans_hold_what_their_launches_read_and_no_more():
    """Device memory of plans: a 1x1 layer has its weights twice where launches of few or many rows read them in operand order, a third
    copy only once it runs behind a depthwise layer; a layer that no such launch comes from has them once."""
    import ctypes as C
    dev = shim.Device()

    def free():
        dev.synchronize()
        left, total = C.c_size_t(), C.c_size_t()
        assert dev.lib.hipMemGetInfo(C.byref(left), C.byref(total)) == 0
        return left.value

    def taken(make):
        make(-1).destroy()                                 # (what the runtime allocates for itself at first)
        before = free()
        keep = [make(k) for k in range(4)]
        used = before - free()
        for p in keep:
            p.destroy()
        return used / 4

    def conv(k, h, ci, co, taps):
        c = cases.make_conv_case("memory", 66000, n=1, h=2, w=2, ci=ci, co=co, kh=taps, kw=taps, in_dtype=U8, in_offset=3, out_offset=0)
        from armnn_amd.tensor import TensorInfo
        xin, yout = (TensorInfo((1, h, h, n), U8, (0.0235,), 3) for n in (ci, co))
        return shim.Conv2dPlan(xin, c.w, c.b, yout, pad_top=taps // 2, pad_left=taps // 2)
    twice = taken(lambda k: conv(k, 28, 768, 8192, 1)) / (768 * 8192)
    once = [taken(lambda k: conv(k, 28, 1024, 8192, 1)) / (1024 * 8192), taken(lambda k: conv(k, 224, 1024, 1024, 3)) / (9 * 1024 * 1024)]
    print(f"times the weights: {twice:.2f}, {once}", flush=True)
    assert twice < 2.6 and max(once) < 1.6
