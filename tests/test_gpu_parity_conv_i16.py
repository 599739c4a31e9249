"""INT16 x INT8 -> INT48 CONV2D on the matrix cores: the 64-channel tiles, K split over one, two and four waves with ragged
shares, channel vectors that are padded, tiles of one pixel or channel, extreme values."""
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


CASES = [  # n, h, w, ic, oc, k, pad, stride, dilation
    (1, 16, 16, 16, 33, 3, 1, 1, 1),     # split 4 in shares of 2, 2, 1 and 0 steps
    (1, 19, 21, 48, 64, 3, 1, 1, 1),     # 27 chunks: the last step is half empty
    (2, 65, 65, 16, 130, 2, 0, 1, 1),    # 64 channels to a wave, ragged both ways
    (1, 130, 130, 32, 24, 1, 0, 1, 1),   # split 1 ... 2 for one or two steps
    (3, 33, 31, 16, 96, 3, 1, 2, 1),
    (1, 20, 20, 32, 40, 3, 2, 1, 2),
    (1, 30, 30, 5, 40, 3, 1, 1, 1),      # channels padded to 16
    (1, 12, 12, 41, 70, 3, 1, 1, 1),     # to 48
]


@pytest.mark.parametrize("case", CASES)
@pytest.mark.parametrize("extreme", [False, True])
def test_conv2d_int16_on_the_matrix_cores(ctx, case, extreme):
    n, h, w, ic, oc, k, p, s, d = case
    rng = np.random.default_rng(ic * oc)
    if extreme:
        x = rng.choice(np.array([-32768, -32641, -129, -128, -1, 0, 127, 128, 32639, 32767], np.int16), (n, h, w, ic))
        wt = rng.choice(np.array([-128, 127], np.int8), (oc, k, k, ic))
    else:
        x = rng.integers(-32768, 32768, (n, h, w, ic)).astype(np.int16)
        wt = rng.integers(-128, 128, (oc, k, k, ic)).astype(np.int8)
    bias = rng.integers(-(1 << 46), 1 << 46, oc).astype(np.int64)
    reach = (k - 1) * d
    pad = (p, p - (h - 1 + 2 * p - reach) % s, p, p - (w - 1 + 2 * p - reach) % s)
    got, st = gpu_ops.conv2d(ctx, x, wt, bias, pad, (s, s), (d, d))
    assert st == capi.VALID and ctx.last_kernel == "conv2d_mfma_i16_i48"
    assert np.array_equal(got, oracle.conv2d("i16", x, wt, bias, pad, (s, s), (d, d)))
