"""DEPTHWISE_CONV2D that walks down the rows: 3x3 and 5x5 taps, strides 1 and 2, channels that are no multiple of four, strips of one row and of
several, every result type, shifts below 32 and values out of their range."""
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


CASES = [  # n, ih, iw, c, k, pads, stride
    (1, 5, 7, 1, 3, (1, 1, 1, 1), 1),
    (2, 9, 8, 7, 3, (1, 1, 1, 1), 1),
    (1, 11, 9, 6, 3, (0, 0, 2, 0), 2),
    (3, 6, 5, 29, 5, (2, 2, 2, 2), 1),
    (1, 13, 12, 30, 5, (1, 1, 2, 1), 2),
    (2, 10, 9, 16, 5, (2, 2, 2, 2), 1),
    (1, 12, 12, 8, 5, (2, 1, 1, 2), 2),
    (1, 3, 3, 5, 3, (0, 0, 0, 0), 1),            # one result
    (20, 61, 61, 61, 3, (1, 1, 1, 1), 1),        # strips of several rows, the last one short
    (9, 75, 70, 44, 5, (2, 2, 2, 2), 1),
    (12, 117, 95, 42, 3, (1, 1, 1, 1), 2),
    (12, 99, 95, 36, 5, (2, 2, 2, 2), 2),
    (8, 60, 60, 44, 3, (1, 1, 1, 1), 1),         # whole groups, 3x3
    (3, 79, 63, 28, 3, (1, 1, 1, 1), 2),
]


@pytest.mark.parametrize("case", CASES)
@pytest.mark.parametrize("in_zp", [0, -128, 9])
def test_depthwise_rows(ctx, case, in_zp):
    n, ih, iw, c, k, pad, s = case
    rng = np.random.default_rng(c * k + ih)
    x, w = rng.integers(-128, 128, (n, ih, iw, c)).astype(np.int8), rng.integers(-128, 128, (k, k, c, 1)).astype(np.int8)
    bias = rng.integers(-9999, 9999, c if c % 3 else 1).astype(np.int32)
    got, st = gpu_ops.conv2d(ctx, x, w, bias, pad, (s, s), in_zp=in_zp, depthwise=True)
    assert st == capi.VALID and ctx.last_kernel == "depthwise_rows_i8"
    want = oracle.depthwise_conv2d("i8", x[-2:], w, np.broadcast_to(bias, c), pad, (s, s), in_zp=in_zp, w_zp=0)
    assert np.array_equal(got[-2:], want)
    if n > 2:
        assert np.array_equal(got[:1], oracle.depthwise_conv2d("i8", x[:1], w, np.broadcast_to(bias, c), pad, (s, s), in_zp=in_zp, w_zp=0))


@pytest.mark.parametrize("case", [CASES[1], CASES[3], CASES[4], CASES[5], CASES[12]])
@pytest.mark.parametrize("shifts", [(34, 40), (31, 33), (20, 28)])    # (the last: values out of the scale's range)
@pytest.mark.parametrize("out_dtype, mode", [(np.int8, capi.ROUND_DOUBLE), (np.int8, capi.ROUND_SINGLE), (np.int16, capi.ROUND_DOUBLE)])
def test_depthwise_rows_fused_rescale(ctx, case, shifts, out_dtype, mode):
    n, ih, iw, c, k, pad, s = case
    rng = np.random.default_rng(c + k + shifts[0])
    span = 128 if shifts[0] > 30 else 8
    x, w = rng.integers(-span, span, (n, ih, iw, c)).astype(np.int8), rng.integers(-span, span, (k, k, c, 1)).astype(np.int8)
    bias = rng.integers(-99, 99, c).astype(np.int32)
    mult, shift = rng.integers(1 << 30, 1 << 31, c).astype(np.int32), rng.integers(*shifts, c).astype(np.int8)
    out_zp, clamp = (-5, (-100, 110)) if out_dtype == np.int8 else (0, None)
    got, st = gpu_ops.conv2d(ctx, x, w, bias, pad, (s, s), in_zp=3, depthwise=True, clamp=clamp,
                             rescale=dict(mult=mult, shift=shift, out_zp=out_zp, out_dtype=out_dtype, rounding_mode=mode))
    assert ctx.last_kernel == "depthwise_rows_i8_rescale"
    acc = oracle.depthwise_conv2d("i8", x, w, bias, pad, (s, s), in_zp=3, w_zp=0)
    want, wst = oracle.rescale(acc, mult, shift, out_zp=out_zp, out_dtype=out_dtype, rounding_mode=mode)
    assert st == wst
    if wst == capi.VALID:
        assert np.array_equal(got, oracle.clamp(want, *clamp) if clamp else want)
