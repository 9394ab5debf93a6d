"""The requantization's fast path over every sum a layer can meet, against the reference's own sequence (a division per value).

A value's bytes come from a bracket around the reference's fp32 value and, where the bracket does not close, from that sequence.
With two channels of full-range codes and weights 127 and 1 the sums of a 1x1 layer are all the integers of a range, so that
each channel's scale and bias meet each of them."""
import numpy as np
import pytest

from armnn_amd import peaks, shim
from armnn_amd.tensor import DataType, QTensor, TensorInfo

pytestmark = pytest.mark.gpu
S8, U8 = DataType.QAsymmS8, DataType.QAsymmU8


def _fast_and_exact(run):
    fast = run()
    shim.set_option("exact_division_epilogue", 1)
    try:
        exact = run()
    finally:
        shim.set_option("exact_division_epilogue", 0)
    return fast, exact


def _scales(kind, channels):
    rng = np.random.default_rng(7)
    if kind == "general":
        return rng.uniform(0.002, 0.02, channels)
    if kind == "powers_of_two":             # sums sit exactly on half-integers
        return 2.0 ** -rng.integers(4, 12, channels)
    if kind == "ratios":                    # ... now and then
        return rng.choice([0.047, 0.02, 0.0235, 0.01], channels) / rng.choice([1, 2, 3, 8], channels)
    if kind == "steps_of_codes":            # a code and more per step of the sum
        return rng.uniform(0.05, 40.0, channels)
    return rng.uniform(1e-9, 1e-7, channels)    # one code for all sums


def test_the_conversion_is_exact_for_every_float():
    """The bracket has no term for v_cvt_pknorm_u16_f32: it has to be rint(65535 x), saturated, for all 2^32 floats but NaN."""
    shim.Device()
    wrong, example = peaks.pknorm_mismatches()
    assert wrong == 0, f"{wrong} floats, {example:#010x} among them"


@pytest.mark.parametrize("clamp", [False, True], ids=["type_range", "clamp_inside"])
@pytest.mark.parametrize("out", [(S8, -128), (U8, 3), (S8, 21)], ids=["s8", "u8", "s8_offset"])
@pytest.mark.parametrize("kind", ["general", "powers_of_two", "ratios", "steps_of_codes", "one_code"])
@pytest.mark.parametrize("ci", [16, 32, 256])
def test_every_sum_of_a_range(kind, ci, out, clamp):
    channels = 64
    codes = np.arange(-128, 128, dtype=np.int8)
    x = np.zeros((1, 256, 256, ci), np.int8)
    x[0, :, :, 0], x[0, :, :, 1] = codes[:, None], codes[None, :]
    w = np.zeros((channels, 1, 1, ci), np.int8)
    w[:, 0, 0, 0], w[:, 0, 0, 1] = 127, 1
    scales = _scales(kind, channels).astype(np.float32)
    b = np.random.default_rng(11).integers(-9000, 9000, channels).astype(np.int32)
    b[::5] = 0
    xq = QTensor(TensorInfo(x.shape, S8, (0.5,), 0), x)
    wq = QTensor(TensorInfo(w.shape, DataType.QSymmS8, tuple(scales), 0, 0), w)
    bq = QTensor(TensorInfo((channels,), DataType.Signed32, tuple(np.float32(0.5) * scales), 0, 0), b)
    info = TensorInfo((1, 256, 256, channels), out[0], (0.25,), out[1])
    act = dict(activation=shim.ACT_BOUNDED_RELU, act_a=20.0, act_b=-1.5) if clamp else {}
    fast, exact = _fast_and_exact(lambda: shim.conv2d(xq, wq, bq, info, **act).data)
    print(f"{kind} {ci}: {shim.last_kernel()}, {len(np.unique(exact))} codes", flush=True)
    np.testing.assert_array_equal(fast, exact)


@pytest.mark.parametrize("scale", [1e-6, 2e-5, 6.2e-5, 1e-4, 3e-3])
@pytest.mark.parametrize("m", [1, 40, 300])
def test_sums_beyond_two_to_the_22nd(m, scale):
    """Sums up to 1.3e8, where the bits of a raised accumulator no longer step in ones; with the small scales codes there are not
    saturated, and the sums are converted."""
    k, o = 4096, 128
    rng = np.random.default_rng(m)
    # rows whose codes and channels whose weights lean to one side more or less: sums of every size
    x = np.clip(rng.integers(-128, 128, (m, k)) + np.linspace(-255, 255, m)[:, None], -128, 127).astype(np.int8)
    w = np.clip(rng.integers(-127, 128, (o, k)) + np.linspace(-254, 254, o)[:, None], -127, 127).astype(np.int8)
    scales = np.full(o, scale, np.float32) * np.linspace(0.5, 1.5, o).astype(np.float32)
    xq = QTensor(TensorInfo((m, k), S8, (1.0,), -3), x)
    wq = QTensor(TensorInfo((o, k), DataType.QSymmS8, tuple(scales), 0, 0), w)
    bq = QTensor(TensorInfo((o,), DataType.Signed32, tuple(scales), 0, 0), rng.integers(-90000, 90000, o).astype(np.int32))
    info = TensorInfo((m, o), S8, (1.0,), 5)
    fast, exact = _fast_and_exact(lambda: shim.fully_connected(xq, wq, bq, info).data)
    print(f"{m} rows, scale {scale}: {shim.last_kernel()}, {len(np.unique(exact))} codes", flush=True)
    np.testing.assert_array_equal(fast, exact)


@pytest.mark.parametrize("m", [1, 40, 300])
def test_sums_beyond_two_to_the_22nd_of_channels_with_the_smallest_scale(m):
    """Such a channel's values are its bias, here a half-integer number of codes, so that all of them are settled one by one, from
    accumulators whose bits are not the sum.  The other channels are saturated beyond 2^22."""
    k, o = 4096, 128
    rng = np.random.default_rng(m)
    x = np.clip(rng.integers(-128, 128, (m, k)) + np.linspace(-255, 255, m)[:, None], -128, 127).astype(np.int8)
    w = np.clip(rng.integers(-127, 128, (o, k)) + np.linspace(-254, 254, o)[:, None], -127, 127).astype(np.int8)
    scales = np.full(o, 3e-3, np.float32)
    scales[::2] = np.float32(1.2e-38)
    b = rng.integers(-260, 260, o).astype(np.int32) * 2 + 1
    xq = QTensor(TensorInfo((m, k), S8, (1.0,), -3), x)
    wq = QTensor(TensorInfo((o, k), DataType.QSymmS8, tuple(scales), 0, 0), w)
    bq = QTensor(TensorInfo((o,), DataType.Signed32, (0.5,) * o, 0, 0), b)
    info = TensorInfo((m, o), S8, (1.0,), 5)
    fast, exact = _fast_and_exact(lambda: shim.fully_connected(xq, wq, bq, info).data)
    print(f"{m} rows: {shim.last_kernel()}, {len(np.unique(exact))} codes", flush=True)
    np.testing.assert_array_equal(fast, exact)


@pytest.mark.parametrize("layer", ["conv1x1", "conv3x3", "depthwise", "classifier", "few_rows", "stem"])
@pytest.mark.parametrize("odd", ["no_weights", "smallest_scale", "always_least", "always_most", "wide", "no_fast_path"])
def test_an_odd_channel_among_others(odd, layer):
    """Channels 5 and 40 are dead, saturated, uncertain over many codes or outside the fast path; the others are as usual."""
    n, h, ci, co, k = {"conv1x1": (2, 28, 64, 128, 1), "conv3x3": (2, 20, 64, 64, 3), "depthwise": (2, 30, 64, 64, 3),
                       "classifier": (1, 40, 1024, 72, 1), "few_rows": (1, 1, 512, 64, 1), "stem": (1, 33, 3, 64, 3)}[layer]
    dw = layer == "depthwise"
    rng = np.random.default_rng(17)
    taps = k * k * (1 if dw else ci)
    w = np.clip(np.rint(rng.standard_normal((1, k, k, co) if dw else (co, k, k, ci)) * 30), -127, 127).astype(np.int8)
    scales = (rng.uniform(0.002, 0.02, co) / np.sqrt(taps) * 3).astype(np.float32)
    b = np.rint(rng.standard_normal(co) * 500).astype(np.int32)
    for c in (5, 40):
        if odd == "no_weights":
            (w[..., c] if dw else w[c])[...] = 0
            scales[c], b[c] = 1.2e-38, 2 ** 31 - 1
        elif odd == "smallest_scale":
            scales[c], b[c] = 1.2e-38, 3
        elif odd == "always_least":
            b[c] = int(-3e4 / scales[c])
        elif odd == "always_most":
            b[c] = int(3e4 / scales[c])
        elif odd == "wide":                       # a bias that some sums take back
            scales[c], b[c] = 0.4, int(-0.3 * 127 * 64 * np.sqrt(taps))
        else:                                     # sums of more codes than the fast path allows
            scales[c], b[c] = 3e7, 12
    stride = 2 if layer == "stem" else 1
    ho = -(-h // stride)
    xq = QTensor(TensorInfo((n, h, h, ci), S8, (0.0235,), -3), rng.integers(-128, 128, (n, h, h, ci)).astype(np.int8))
    wq = QTensor(TensorInfo(w.shape, DataType.QSymmS8, tuple(scales), 0, 3 if dw else 0), w)
    bq = QTensor(TensorInfo((co,), DataType.Signed32, tuple(np.float32(0.0235) * scales), 0, 0), b)
    info = TensorInfo((n, ho, ho, co), S8, (0.0235,), -20)
    fast, exact = _fast_and_exact(lambda: shim.conv2d(xq, wq, bq, info, pad_top=k // 2, pad_left=k // 2, stride_x=stride, stride_y=stride, depthwise=dw).data)
    print(f"{odd} {layer}: {shim.last_kernel()}, {len(np.unique(exact))} codes, of channel 5 {len(np.unique(exact[..., 5]))}", flush=True)
    np.testing.assert_array_equal(fast, exact)
