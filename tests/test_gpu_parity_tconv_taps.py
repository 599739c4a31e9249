"""TRANSPOSE_CONV2D class by class of output pixels: strides of two to four, one tap of a class and several, cropped and padded outputs, channels of
no whole chunks, the last bytes of both operands, one, two and four channel tiles, several tiles to a wave."""
import numpy as np
import pytest

import gpu_ops
import oracle
from reference_model_amd import Context, capi

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = Context(0)
    yield c
    c.close()


CASES = [  # n, ih, iw, ic, oc, kh, kw, out_pad, stride
    (1, 7, 9, 16, 17, 2, 2, (0, 0, 0, 0), (2, 2)),         # a tap to a class
    (2, 9, 11, 48, 16, 3, 3, (0, -1, 0, -1), (2, 2)),      # one, two and four
    (1, 6, 5, 24, 33, 4, 4, (-1, -1, -1, -1), (2, 2)),     # cropped
    (2, 5, 6, 20, 70, 5, 4, (1, 0, 0, 2), (2, 2)),         # out beyond the input
    (1, 8, 7, 33, 9, 3, 5, (0, 0, -1, -1), (3, 2)),        # strides of their own
    (1, 5, 9, 7, 40, 1, 4, (0, 0, 0, 0), (1, 4)),
    (1, 6, 6, 65, 64, 7, 3, (-2, -1, 0, 0), (4, 3)),
    (3, 13, 12, 32, 128, 4, 4, (-1, -1, -1, -1), (2, 2)),  # two and four channel tiles
    (4, 40, 40, 40, 60, 2, 2, (0, 0, 0, 0), (2, 2)),
    (2, 90, 91, 16, 12, 3, 3, (0, -1, 0, -1), (2, 2)),     # several tiles to a wave
    (1, 4, 4, 272, 24, 3, 3, (0, -1, 0, -1), (2, 2)),      # 68 chunks
    (1, 1, 1, 17, 5, 2, 2, (0, 0, 0, 0), (2, 2)),          # one input pixel
    (2, 9, 7, 26, 20, 3, 3, (0, 0, 0, 0), (2, 2)),         # classes of different sizes
    (1, 5, 5, 8, 8, 3, 4, (0, -2, 1, 0), (3, 4)),
]


@pytest.mark.parametrize("case", CASES)
@pytest.mark.parametrize("in_zp", [0, -7, 127])
def test_transpose_conv2d_by_classes(ctx, case, in_zp):
    n, ih, iw, ic, oc, kh, kw, out_pad, stride = case
    rng = np.random.default_rng(ic * oc + kh)
    x, w = (rng.integers(-128, 128, s).astype(np.int8) for s in ((n, ih, iw, ic), (oc, kh, kw, ic)))
    for bias in (rng.integers(-9999, 9999, oc).astype(np.int32), np.array([77], np.int32)):
        got, st = gpu_ops.transpose_conv2d(ctx, x, w, bias, out_pad, stride, in_zp, 0)
        assert st == capi.VALID and ctx.last_kernel == "transpose_conv2d_taps_i8"
        assert np.array_equal(got, oracle.transpose_conv2d("i8", x, w, bias, out_pad, stride, in_zp, 0))
