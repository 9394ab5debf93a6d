"""One to four rows of a FullyConnected or 1x1 layer (a matrix-vector kernel) against the plain kernel, bit for bit: K of one piece of 16
bytes up to several rounds of four steps, ends inside a step, channel counts that are no multiple of a lane's four, a wave's or a
block's, weights with a zero point."""
import numpy as np
import pytest

from armnn_amd import shim
from tests import cases

pytestmark = pytest.mark.gpu
U8, S8 = cases.U8, cases.S8


@pytest.mark.parametrize("zw", [0, 93], ids=["symmetric", "zero_point"])
@pytest.mark.parametrize("k,o", [(16, 1), (16, 130), (1008, 3), (1024, 16), (1040, 129), (2032, 21), (3088, 257), (4096, 64), (5136, 5), (9216, 40)])
@pytest.mark.parametrize("m", [1, 2, 3, 4])
def test_few_rows_of_a_matrix(m, k, o, zw):
    dt = U8 if (k // 16 + m) % 2 else S8
    wq = dict(w_dtype=U8, w_offset=zw, per_axis=False) if zw else {}
    c = cases.make_conv_case("gemv", 91000 + k + 7 * m + zw, n=1, h=1, w=m, ci=k, co=o, kh=1, kw=1, in_dtype=dt, in_scale=0.0235,
                             in_offset=121 if dt == U8 else -7, out_scale=0.1, out_offset=100 if dt == U8 else -20, **wq)
    got = shim.conv2d(c.x, c.w, c.b, c.out_info, **c.params)
    kernel = shim.last_kernel()
    print(m, k, o, kernel, flush=True)
    assert kernel == f"GemvKernel<{min(m, 2)}>", kernel
    np.testing.assert_array_equal(got.data, shim.conv2d(c.x, c.w, c.b, c.out_info, algo=shim.ALGO_DIRECT, **c.params).data)
