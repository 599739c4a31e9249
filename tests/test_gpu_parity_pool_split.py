"""Integer pooling with the taps of a window dealt over 16 lanes: windows of 16 taps and more, cut by the border and not, with
ragged numbers of taps, channel groups and results."""
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


@pytest.mark.parametrize("dtype", [np.int8, np.int16])
@pytest.mark.parametrize("case", [  # n, h, w, c, kernel, stride, pad
    (1, 7, 7, 16, (7, 7), (7, 7), (0, 0, 0, 0)), (3, 4, 4, 48, (4, 4), (1, 1), (0, 0, 0, 0)), (2, 9, 11, 80, (5, 5), (2, 2), (2, 2, 2, 2)),
    (5, 13, 5, 32, (13, 5), (13, 5), (0, 0, 0, 0)), (1, 40, 33, 16, (40, 33), (1, 1), (0, 0, 0, 0)), (2, 8, 8, 16, (2, 9), (1, 1), (1, 1, 4, 4))])
def test_windows_over_sixteen_lanes(ctx, dtype, case):
    n, h, w, c, k, s, p = case
    rng = np.random.default_rng(h * w + c)
    info = np.iinfo(dtype)
    x = rng.integers(info.min, info.max + 1, (n, h, w, c)).astype(dtype)
    zps = (-7, 5) if dtype == np.int8 else (0, 0)
    got, st = gpu_ops.pool2d(ctx, x, k, s, p, True, *zps)
    assert ctx.last_kernel == ("avg_pool2d_split_i8" if dtype == np.int8 else "avg_pool2d_split_i16")
    assert st == capi.VALID and np.array_equal(got, oracle.avg_pool2d(x, k, s, p, *zps))
    got, st = gpu_ops.pool2d(ctx, x, k, s, p, False)
    assert ctx.last_kernel == ("max_pool2d_split_i8" if dtype == np.int8 else "max_pool2d_split_i16")
    assert st == capi.VALID and np.array_equal(got, oracle.max_pool2d(x, k, s, p))
