"""1x1 layers and FullyConnected whose channels end inside a 128-byte k-tile, on the direct-to-LDS kernels, against the plain kernel,
bit for bit: one and seven 16-byte pieces in the last tile, ragged rows and output channels, weights with a zero point."""
import numpy as np
import pytest

from armnn_amd import shim
from tests import cases

pytestmark = pytest.mark.gpu
U8, S8 = cases.U8, cases.S8

LAYERS = [
    (1500, 912, 304, "IgemmLdsKernel<64, 64, 2, 2, 3"),
    (1999, 1008, 640, "IgemmLdsKernel<64, 64, 2, 2, 2"),
    (6401, 1040, 1030, "BigGemmKernel<256, 128, 3"),
    (5200, 784, 1200, "IgemmLdsKernel<128, 128, 2, 2, 2"),
    (8190, 1296, 2048, "BigGemmKernel<256, 256, 2"),
    (2537, 1712, 3548, "IgemmKernel<128, 128, 2, 2, 2, 64"),
]


@pytest.mark.parametrize("zw", [0, 93], ids=["symmetric", "zero_point"])
@pytest.mark.parametrize("m,k,o,name", LAYERS, ids=[f"{l[0]}x{l[1]}_{l[2]}" for l in LAYERS])
def test_last_k_tile_ends_early(m, k, o, name, zw):
    dt = U8 if k // 16 % 2 else S8
    wq = dict(w_dtype=U8, w_offset=zw, per_axis=False) if zw else {}
    c = cases.make_conv_case("tail", 81000 + k + zw, n=1, h=1, w=m, ci=k, co=o, kh=1, kw=1, in_dtype=dt, in_scale=0.0235,
                             in_offset=121 if dt == U8 else -7, out_scale=0.1, out_offset=100 if dt == U8 else -20, **wq)
    got = shim.conv2d(c.x, c.w, c.b, c.out_info, **c.params)
    kernel = shim.last_kernel()
    print(kernel, flush=True)
    assert kernel.startswith(name) and (kernel.endswith("true>") or name.startswith("IgemmKernel")), kernel
    assert len(np.unique(got.data)) > 8
    np.testing.assert_array_equal(got.data, shim.conv2d(c.x, c.w, c.b, c.out_info, algo=shim.ALGO_DIRECT, **c.params).data)
