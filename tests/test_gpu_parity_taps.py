"""CONV2D with resident weights or a split reduction, operands read as they lie (conv_taps.hip): the sizes where a tile, a chunk of the
channel vector, the last bytes of a tensor or a store can go wrong.  Integers bit for bit against the oracle; fp16 and bf16 against
fp64 on values whose sums are exact in fp32, so that one rounding of the result is all there is."""
import numpy as np
import pytest

import gpu_ops
import oracle
from reference_model_amd import Context, capi

pytestmark = pytest.mark.gpu

# n, h, w, ic, oc, (kh, kw), (top, bottom, left, right), (sy, sx), (dy, dx)
SPLIT = [  # at most a workgroup's tile of 32 x 32 results per slot: the reduction is split
    (1, 9, 23, 8, 44, (3, 3), (1, 1, 1, 1), (1, 1), (1, 1)),          # half a chunk a tap, an odd count of chunks
    (2, 17, 19, 24, 100, (3, 5), (1, 1, 0, 4), (1, 1), (1, 1)),       # a chunk and a half; uneven pads; odd last tiles of pixels and channels
    (3, 14, 15, 200, 43, (3, 3), (1, 1, 1, 1), (1, 1), (1, 1)),       # 59 steps: eight waves, several groups of steps
    (1, 40, 31, 40, 9, (1, 1), (0, 0, 0, 0), (1, 1), (1, 1)),         # one tap; channels by ones
    (2, 15, 15, 48, 130, (2, 3), (0, 1, 2, 0), (2, 2), (1, 1)),       # strides
    (1, 33, 35, 36, 20, (3, 3), (2, 2, 2, 2), (1, 1), (2, 2)),        # dilation; words but no pieces of 16 bytes
    (5, 16, 17, 13, 33, (3, 3), (1, 1, 1, 1), (1, 1), (1, 1)),        # odd addresses; the tensor ends inside a chunk
    (20, 13, 13, 304, 45, (3, 3), (0, 0, 0, 0), (2, 2), (1, 1)),      # 86 steps
]
MANY = [  # many tiles: weights resident, one to four channel tiles a wave
    (7, 61, 59, 16, 30, (3, 3), (1, 1, 1, 1), (1, 1), (1, 1)),
    (5, 70, 71, 20, 101, (1, 1), (0, 0, 0, 0), (1, 1), (1, 1)),       # channels by ones: rows gathered in LDS
    (9, 64, 62, 7, 84, (3, 3), (1, 1, 1, 1), (1, 1), (1, 1)),         # odd addresses; 84 = three channel tiles, the last part empty
    (8, 55, 57, 12, 66, (3, 3), (1, 1, 1, 1), (1, 1), (1, 1)),
    (6, 90, 88, 16, 250, (1, 2), (0, 0, 1, 0), (1, 1), (1, 1)),       # several channel blocks, channels by twos
]


@pytest.fixture(scope="module")
def ctx():
    c = Context(0)
    yield c
    c.close()


def _fitting(case):
    """the case with the bottom and right pads a whole number of steps needs"""
    n, h, w, ic, oc, k, pad, stride, dil = case
    pad = list(pad)
    for axis, size in ((0, h), (1, w)):
        full = size - 1 + pad[2 * axis] + pad[2 * axis + 1] - (k[axis] - 1) * dil[axis]
        pad[2 * axis + 1] += -full % stride[axis]
    return n, h, w, ic, oc, k, tuple(pad), stride, dil


@pytest.mark.parametrize("case", SPLIT + MANY)
@pytest.mark.parametrize("form", ["int32", "int8", "relu", "small shifts", "int16"])
def test_int8(ctx, case, form):
    n, h, w, ic, oc, k, pad, stride, dil = _fitting(case)
    rng = np.random.default_rng(ic * oc)
    x, wt = rng.integers(-128, 128, (n, h, w, ic)).astype(np.int8), rng.integers(-128, 128, (oc, *k, ic)).astype(np.int8)
    bias = rng.integers(-9999, 9999, oc).astype(np.int32)
    want = oracle.conv2d("i8", x, wt, bias, pad, stride, dil, in_zp=-11, w_zp=0)
    if form == "int32":
        got, st = gpu_ops.conv2d(ctx, x, wt, bias, pad, stride, dil, in_zp=-11, w_zp=0)
        assert st == capi.VALID and np.array_equal(got, want) and ctx.last_kernel == "conv2d_taps_i8"
        return
    reach = k[0] * k[1] * ic
    base = 38 + int(np.log2(reach)) // 2 - (8 if form == "int16" else 0)
    mult, shift = rng.integers(1 << 30, 1 << 31, oc).astype(np.int32), rng.integers(base, base + 3, oc).astype(np.int8)
    if form == "small shifts":      # the general form of the rescale; every value legal: |v| < 2^30
        mult, shift = rng.integers(1 << 15, 1 << 16, oc).astype(np.int32), rng.integers(22, 32, oc).astype(np.int8)
    out = np.int16 if form == "int16" else np.int8
    zp = 0 if form == "int16" else 3
    rescale = dict(mult=mult, shift=shift, out_zp=zp, out_dtype=out, rounding_mode=capi.ROUND_SINGLE if form == "relu" else capi.ROUND_DOUBLE)
    clamp = (3, 90) if form == "relu" else None
    want, wst = oracle.rescale(want, mult, shift, out_zp=zp, out_dtype=out, rounding_mode=rescale["rounding_mode"])
    if clamp:
        want = np.clip(want, *clamp)
    got, st = gpu_ops.conv2d(ctx, x, wt, bias, pad, stride, dil, in_zp=-11, w_zp=0, rescale=rescale, clamp=clamp)
    assert st == wst and np.array_equal(got, want) and len(np.unique(got)) > 20 and ctx.last_kernel == "conv2d_taps_i8_rescale"


@pytest.mark.parametrize("case", SPLIT + MANY)
@pytest.mark.parametrize("dtype", [capi.FP16, capi.BF16])
def test_16_bit_floats(ctx, case, dtype):
    n, h, w, ic, oc, k, pad, stride, dil = _fitting(case)
    rng = np.random.default_rng(ic * oc)
    # whole quarters: exact in both types, and so are the products and the sums of a few thousand of them in fp32
    x, wt, bias = (rng.integers(-8, 9, sh).astype(np.float32) / 4 for sh in ((n, h, w, ic), (oc, *k, ic), (oc,)))
    want = oracle.conv2d("f64", *(v.astype(np.float64) for v in (x, wt, bias)), pad, stride, dil)
    if dtype == capi.FP16:
        args = [v.astype(np.float16) for v in (x, wt, bias)]
    else:
        args = [(v.view(np.uint32) >> 16).astype(np.uint16) for v in (x, wt, bias)]
    got, st = gpu_ops.conv2d(ctx, *args, pad, stride, dil, dtype=dtype)
    assert st == capi.VALID and ctx.last_kernel == ("conv2d_taps_f16" if dtype == capi.FP16 else "conv2d_taps_bf16")
    if dtype == capi.BF16:
        got = (got.astype(np.uint32) << 16).view(np.float32)
    ulp = 2.0 ** -11 if dtype == capi.FP16 else 2.0 ** -8
    assert np.all(np.abs(got.astype(np.float64) - want) <= ulp * np.abs(want))


@pytest.mark.parametrize("dtype", [capi.FP16, capi.BF16])
@pytest.mark.parametrize("shape", [(2, 20, 21, 9, 40), (9, 50, 50, 6, 33)])
def test_infinities_stay_where_they_are(ctx, dtype, shape):
    """an infinite channel reaches the results whose windows hold it and no other, although a chunk reads past its channel vector"""
    n, h, w, ic, oc = shape
    rng = np.random.default_rng(4)
    x, wt, bias = rng.normal(size=(n, h, w, ic)), rng.uniform(0.5, 1.0, (oc, 3, 3, ic)), np.zeros(oc)
    x[1, 7, 5, 0] = np.inf
    x[0, h - 1, w - 1, ic - 1] = -np.inf
    want = oracle.conv2d("f64", x, wt, bias, (1, 1, 1, 1), (1, 1), (1, 1))
    if dtype == capi.FP16:
        args = [v.astype(np.float16) for v in (x, wt, bias)]
    else:
        args = [(v.astype(np.float32).view(np.uint32) >> 16).astype(np.uint16) for v in (x, wt, bias)]
    got, st = gpu_ops.conv2d(ctx, *args, (1, 1, 1, 1), (1, 1), (1, 1), dtype=dtype)
    got = got.astype(np.float32) if dtype == capi.FP16 else (got.astype(np.uint32) << 16).view(np.float32)
    assert st == capi.VALID and "taps" in ctx.last_kernel
    assert np.array_equal(np.isposinf(got), np.isposinf(want)) and np.array_equal(np.isneginf(got), np.isneginf(want)) and not np.isnan(got).any()


@pytest.mark.parametrize("dtype", [capi.FP16, capi.BF16])
@pytest.mark.parametrize("shape, stride", [
    ((2, 20, 21, 9, 40), 1),       # a split reduction, ragged
    ((1, 9, 23, 8, 44), 1),        # whole pieces
    ((9, 50, 50, 6, 33), 1),       # resident weights; rows gathered in LDS
    ((9, 50, 50, 16, 70), 1),      # several channel tiles a wave
    ((15, 54, 65, 68, 60), 2)])
def test_infinite_weights_under_taps_outside_the_image(ctx, dtype, shape, stride):
    """a tap outside the image adds nothing, whatever its weight; inside, an infinity or a NaN reaches its results"""
    n, h, w, ic, oc = shape
    n, h, w, ic, oc, k, pad, _, _ = _fitting((n, h, w, ic, oc, (3, 3), (1, 1, 1, 1), (stride, stride), (1, 1)))
    rng = np.random.default_rng(6)
    x, wt, bias = (rng.integers(-8, 9, sh).astype(np.float32) / 4 for sh in ((n, h, w, ic), (oc, 3, 3, ic), (oc,)))
    wt[oc // 2, 0, 0, 1], wt[oc - 1, 2, 1, 0], wt[1, 1, 2, ic - 1] = np.inf, np.nan, -np.inf
    x[0, 0, 1, 0] = np.nan
    with np.errstate(invalid="ignore"):
        want = oracle.conv2d("f64", *(v.astype(np.float64) for v in (x, wt, bias)), pad, (stride, stride), (1, 1))
    if dtype == capi.FP16:
        args = [v.astype(np.float16) for v in (x, wt, bias)]
    else:
        args = [(v.view(np.uint32) >> 16).astype(np.uint16) for v in (x, wt, bias)]
    got, st = gpu_ops.conv2d(ctx, *args, pad, (stride, stride), dtype=dtype)
    got = got.astype(np.float64) if dtype == capi.FP16 else (got.astype(np.uint32) << 16).view(np.float32).astype(np.float64)
    assert st == capi.VALID and "taps" in ctx.last_kernel
    assert np.array_equal(np.isnan(got), np.isnan(want)) and np.isinf(want).any() and np.isnan(want).any()
    finite = np.isfinite(want)
    assert np.array_equal(got[~finite], want[~finite], equal_nan=True)
    assert np.all(np.abs(got[finite] - want[finite]) <= (2.0 ** -11 if dtype == capi.FP16 else 2.0 ** -8) * np.abs(want[finite]))


def test_values_out_of_range_are_latched(ctx):
    """apply_scale_32's value range, by stored results only"""
    for shape in ((1, 9, 23, 8, 44), (9, 64, 62, 7, 84)):
        n, h, w, ic, oc = shape
        x, wt = np.full((n, h, w, ic), 127, np.int8), np.full((oc, 3, 3, ic), 127, np.int8)
        bias = np.zeros(oc, np.int32)
        for shift, status in ((30, capi.VALID), (12, capi.UNPREDICTABLE)):
            mult, sh = np.full(oc, 1 << 12, np.int32), np.full(oc, shift, np.int8)
            _, st = gpu_ops.conv2d(ctx, x, wt, bias, (1, 1, 1, 1), in_zp=0, w_zp=0, rescale=dict(mult=mult, shift=sh))
            assert "taps" in ctx.last_kernel and st == status


@pytest.mark.parametrize("shape, form, kernel, copies", [
    ((1, 40, 40, 5, 16), "16-bit scales", "conv2d_direct_i8_rescale", False),     # (this kernel would lead)
    ((1, 40, 40, 3, 16), "off 16 bytes", "conv2d_direct_i8", False),
    ((2, 35, 35, 45, 8), "16-bit scales", "conv2d_mfma_i8_rescale", True),        # rows of no whole words: padded first
    ((2, 35, 35, 45, 8), "off 16 bytes", "conv2d_mfma_i8", True),
    ((18, 21, 21, 48, 16), "16-bit scales", "conv2d_mfma_i8_rescale", False),     # whole words: the patch kernel, as they lie
    ((18, 21, 21, 48, 16), "off 16 bytes", "conv2d_mfma_i8", False)])
def test_what_it_declines_goes_where_it_leads(shape, form, kernel, copies):
    """results off 16 bytes and 16-bit multipliers are not this kernel's: the rules that would hand it such a layer look for the next best"""
    n, h, w, ic, oc = shape
    rng = np.random.default_rng(ic)
    x, wt = rng.integers(-128, 128, (n, h, w, ic)).astype(np.int8), rng.integers(-128, 128, (oc, 3, 3, ic)).astype(np.int8)
    bias = rng.integers(-9999, 9999, oc).astype(np.int32)
    want = oracle.conv2d("i8", x, wt, bias, (1, 1, 1, 1), (1, 1), (1, 1), in_zp=-11, w_zp=0)
    c = Context(0)
    try:
        if form == "16-bit scales":
            mult, shift = rng.integers(1 << 14, 1 << 15, oc).astype(np.int16), rng.integers(22, 25, oc).astype(np.int8)
            r = dict(mult=mult, shift=shift, out_zp=3, scale32=False, rounding_mode=capi.ROUND_SINGLE)
            want, wst = oracle.rescale(want, mult, shift, out_zp=3, scale32=False, rounding_mode=capi.ROUND_SINGLE)
            got, st = gpu_ops.conv2d(c, x, wt, bias, (1, 1, 1, 1), in_zp=-11, w_zp=0, rescale=r)
        else:
            d = c.conv_desc(capi.INT8, capi.INT32, x.shape, oc, 3, 3, (h, w), (1, 1, 1, 1), (1, 1), (1, 1), oc)
            out = c.empty((want.size + 1,), capi.INT32)
            c.conv2d(d, *(c.upload(v) for v in (x, wt, bias)), -11, 0, out.ptr + 4)
            st, wst, got = c.sync(), capi.VALID, out.numpy()[1:].reshape(want.shape)
        assert st == wst and np.array_equal(got, want)
        assert c.last_kernel == kernel and (c.workspace_bytes() != (0, 0)) == copies
    finally:
        c.close()


@pytest.mark.parametrize("dtype, shape, k, kernel", [
    (capi.FP16, (6, 91, 61, 4, 96), 3, "conv2d_mfma_f16"),      # rows of two words, many tiles: not filled up to 16 bytes a tap
    (capi.FP16, (1, 91, 61, 4, 96), 3, "conv2d_taps_f16"),      # fewer than it has workgroups
    (capi.BF16, (7, 51, 60, 6, 56), 5, "conv2d_mfma_bf16"),
    (capi.BF16, (7, 51, 60, 6, 60), 5, "conv2d_taps_bf16"),     # channels by fours
    (capi.FP16, (3, 87, 100, 12, 8), 1, "conv2d_mfma_f16"),
    (capi.FP16, (3, 87, 100, 16, 8), 1, "conv2d_taps_f16"),
    (capi.INT8, (15, 13, 8, 26, 568), 1, "conv2d_pointwise_i8_rescale"),    # on copies
    (capi.INT8, (1, 49, 40, 27, 360), 1, "conv2d_taps_i8_rescale"),
    (capi.INT8, (30, 40, 16, 43, 51), 5, "conv2d_mfma_i8_rescale"),         # on copies of 64 bytes
    (capi.FP16, (8, 60, 60, 10, 64), 7, "conv2d_mfma_f16"),
    (capi.FP16, (20, 84, 32, 14, 4), 7, "conv2d_mfma_f16"),                 # few channels
    (capi.BF16, (45, 29, 27, 4, 1), 11, "conv2d_mfma_bf16"),
    (capi.FP16, (8, 60, 60, 10, 64), 9, "conv2d_taps_f16"),                 # windows whose weights do not fit the patch kernel's LDS
    (capi.FP16, (4, 60, 60, 8, 64), 13, "conv2d_taps_f16"),
    (capi.BF16, (2, 60, 60, 64, 256), 13, "conv2d_taps_bf16"),
    (capi.INT8, (4, 60, 60, 16, 64), 13, "conv2d_taps_i8_rescale")])
def test_many_tiles_of_short_rows_go_where_they_lead(ctx, dtype, shape, k, kernel):
    n, h, w, ic, oc = shape
    rng = np.random.default_rng(ic)
    pad = (k // 2,) * 4
    if dtype == capi.INT8:
        x, wt = rng.integers(-128, 128, (n, h, w, ic)).astype(np.int8), rng.integers(-128, 128, (oc, k, k, ic)).astype(np.int8)
        bias = rng.integers(-9999, 9999, oc).astype(np.int32)
        mult, shift = rng.integers(1 << 30, 1 << 31, oc).astype(np.int32), rng.integers(40, 43, oc).astype(np.int8)
        got, st = gpu_ops.conv2d(ctx, x, wt, bias, pad, in_zp=-11, w_zp=0, rescale=dict(mult=mult, shift=shift, out_zp=3))
        want, wst = oracle.rescale(oracle.conv2d("i8", x[-1:], wt, bias, pad, in_zp=-11, w_zp=0), mult, shift, out_zp=3)
        assert st == wst and np.array_equal(got[-1:], want)
    else:
        x, wt, bias = (rng.integers(-8, 9, s).astype(np.float32) / 4 for s in ((n, h, w, ic), (oc, k, k, ic), (oc,)))
        args = [v.astype(np.float16) if dtype == capi.FP16 else (v.view(np.uint32) >> 16).astype(np.uint16) for v in (x, wt, bias)]
        got, st = gpu_ops.conv2d(ctx, *args, pad, dtype=dtype)
        got = got[-1:].astype(np.float64) if dtype == capi.FP16 else (got[-1:].astype(np.uint32) << 16).view(np.float32).astype(np.float64)
        want = oracle.conv2d("f64", *(v.astype(np.float64) for v in (x[-1:], wt, bias)), pad, (1, 1), (1, 1))
        assert st == capi.VALID and np.all(np.abs(got - want) <= (2.0 ** -11 if dtype == capi.FP16 else 2.0 ** -8) * np.abs(want))
    assert ctx.last_kernel == kernel
