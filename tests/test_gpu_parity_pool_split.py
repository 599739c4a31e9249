"""Integer pooling with the taps of a window dealt over 16 lanes: windows of many taps, cut by the border and not, with ragged
numbers of taps, channel groups and results; and the border to the kernel with a lane per window."""
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
    kernel = "pool2d_vec_i8" if dtype == np.int8 and k[0] * k[1] < 24 else ("pool2d_split_i8" if dtype == np.int8 else "pool2d_split_i16")
    assert ctx.last_kernel == "avg_" + kernel
    assert st == capi.VALID and np.array_equal(got, oracle.avg_pool2d(x, k, s, p, *zps))
    got, st = gpu_ops.pool2d(ctx, x, k, s, p, False)
    assert ctx.last_kernel == "max_" + kernel
    assert st == capi.VALID and np.array_equal(got, oracle.max_pool2d(x, k, s, p))


@pytest.mark.parametrize("dtype, case, kernel", [  # n, h, w, c, kernel and stride
    (np.int8, (2, 8, 8, 64, 4), "vec"), (np.int8, (4, 160, 64, 256, 4), "vec"),          # 16 taps: 32 and 10 240 groups
    (np.int8, (4, 5, 5, 1024, 5), "split"), (np.int8, (4, 50, 50, 256, 5), "vec"),       # 25 taps: 256 and 6400
    (np.int8, (4, 28, 28, 1024, 7), "split"), (np.int8, (4, 112, 112, 256, 7), "vec"),    # 49 taps: 4096 and 16 384
    (np.int16, (2, 8, 8, 64, 4), "split"), (np.int16, (4, 256, 32, 256, 4), "vec"),       # 64 and 16 384 groups of eight channels
])
def test_border_to_the_lane_per_window(ctx, dtype, case, kernel):
    n, h, w, c, k = case
    rng = np.random.default_rng(h + c)
    info = np.iinfo(dtype)
    x = rng.integers(info.min, info.max + 1, (n, h, w, c)).astype(dtype)
    zps = (-7, 5) if dtype == np.int8 else (0, 0)
    suffix = "_i8" if dtype == np.int8 else "_i16"
    got, st = gpu_ops.pool2d(ctx, x, (k, k), (k, k), (0, 0, 0, 0), True, *zps)
    assert st == capi.VALID and ctx.last_kernel == "avg_pool2d_" + kernel + suffix
    assert np.array_equal(got, oracle.avg_pool2d(x, (k, k), (k, k), (0, 0, 0, 0), *zps))
    got, st = gpu_ops.pool2d(ctx, x, (k, k), (k, k), (0, 0, 0, 0), False)
    assert st == capi.VALID and ctx.last_kernel == "max_pool2d_" + kernel + suffix
    assert np.array_equal(got, oracle.max_pool2d(x, (k, k), (k, k), (0, 0, 0, 0)))
