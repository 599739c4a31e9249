"""INT16 x INT8 -> INT48 CONV2D with the weights in LDS: one, two and four channel tiles, K split over the waves of a workgroup or not, channels
of no whole chunks, the last bytes of both operands, several tiles to a wave."""
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


CASES = [  # n, h, w, ic, oc, kh, kw, pads, strides, dilations
    (1, 10, 25, 16, 33, 1, 1, (0, 0, 0, 0), (1, 1), (1, 1)),     # one tile of channels to a workgroup, half a step
    (3, 33, 31, 16, 15, 3, 3, (1, 1, 1, 1), (1, 1), (1, 1)),     # split: shares of one step and none
    (1, 20, 21, 80, 40, 3, 3, (2, 0, 1, 2), (1, 1), (1, 1)),     # 45 chunks, uneven padding
    (1, 103, 38, 16, 130, 2, 2, (1, 0, 1, 0), (2, 1), (1, 1)),   # two tiles, strided
    (1, 54, 38, 16, 20, 3, 3, (2, 2, 2, 2), (1, 1), (2, 2)),     # two tiles, split, dilated
    (4, 60, 60, 16, 64, 3, 3, (1, 1, 1, 1), (1, 1), (1, 1)),     # four tiles
    (5, 90, 91, 32, 21, 1, 1, (0, 0, 0, 0), (1, 1), (1, 1)),     # several tiles of pixels to a wave
    (1, 45, 48, 20, 33, 1, 1, (0, 0, 0, 0), (1, 1), (1, 1)),     # even channels, no padding: the end of the tensor
    (1, 17, 9, 26, 33, 2, 2, (0, 0, 0, 0), (1, 1), (1, 1)),
    (2, 30, 57, 18, 70, 1, 3, (0, 0, 0, 1), (1, 1), (1, 1)),
    (2, 90, 91, 26, 128, 3, 3, (0, 0, 0, 0), (1, 1), (1, 1)),
    (1, 12, 13, 33, 20, 2, 3, (0, 0, 0, 0), (1, 1), (1, 1)),     # odd channels
    (1, 38, 57, 33, 35, 1, 1, (0, 0, 0, 0), (1, 1), (1, 1)),
    (1, 60, 57, 35, 70, 2, 1, (0, 0, 0, 0), (1, 1), (1, 1)),
    (3, 50, 50, 1, 17, 5, 5, (2, 2, 2, 2), (1, 1), (1, 1)),      # one channel
]


@pytest.mark.parametrize("case", CASES)
@pytest.mark.parametrize("extreme", [False, True])
def test_conv2d_int16_with_resident_weights(ctx, case, extreme):
    n, h, w, ic, oc, kh, kw, pad, stride, dil = case
    rng = np.random.default_rng(ic * oc)
    if extreme:
        x = rng.choice(np.array([-32768, -32641, -129, -128, -1, 0, 127, 128, 32639, 32767], np.int16), (n, h, w, ic))
        wt = rng.choice(np.array([-128, 127], np.int8), (oc, kh, kw, ic))
    else:
        x = rng.integers(-32768, 32768, (n, h, w, ic)).astype(np.int16)
        wt = rng.integers(-128, 128, (oc, kh, kw, ic)).astype(np.int8)
    bias = rng.integers(-(1 << 46), 1 << 46, 1 if ic == 16 else oc).astype(np.int64)
    got, st = gpu_ops.conv2d(ctx, x, wt, bias, pad, stride, dil)
    assert st == capi.VALID and ctx.last_kernel == "conv2d_mfma_i16_i48"
    assert np.array_equal(got, oracle.conv2d("i16", x, wt, np.broadcast_to(bias, oc), pad, stride, dil))
