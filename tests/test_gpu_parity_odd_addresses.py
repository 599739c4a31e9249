"""Operands on addresses of no alignment although their channel vectors are whole pieces: the forms of the kernels that stream pixels past
resident weights, and of the one that walks down the rows, that read such operands.  What lies around an operand - the largest values,
infinities - reaches no result."""
import numpy as np
import pytest

import oracle
from reference_model_amd import Context, capi

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = Context(0)
    yield c
    for p in list(c._owned):
        c._free(p)
    c.close()


def _put(ctx, v, off):
    """v in the middle of a buffer of its type's infinity (integers: all bits of a byte but the sign), `off` bytes off 256"""
    around = np.full(64, 0x7C00, np.uint16) if v.dtype == np.float16 else (np.full(64, 0x7F80, np.uint16) if v.dtype == np.uint16 else np.full(128, 0x7F, np.uint8))
    around = around.view(np.uint8)
    raw    = np.concatenate([np.resize(around, off), np.ascontiguousarray(v).ravel().view(np.uint8), around])
    return ctx.upload(raw, capi.INT8).ptr + off


def _conv_desc(ctx, in_dtype, out_dtype, x, oc, k, stride):
    n, h, w, _ = x.shape
    oh, ow = (h + 2 * (k // 2) - k) // stride + 1, (w + 2 * (k // 2) - k) // stride + 1
    return ctx.conv_desc(in_dtype, out_dtype, x.shape, oc, k, k, (oh, ow), (k // 2,) * 4, (stride, stride), (1, 1), oc), (n, oh, ow, oc)


OFFSETS = [(1, 0), (0, 1), (4, 12), (8, 4), (15, 3)]    # in, weights; in bytes, doubled for elements of two
CONV = [  # n, h, w, ic, oc, k, stride: the reduction split, weights resident; one and several channel tiles
    (1, 9, 11, 16, 44, 3, 1), (2, 15, 15, 48, 32, 3, 2), (1, 13, 13, 304, 45, 3, 1),
    (7, 61, 59, 16, 30, 3, 1), (9, 64, 62, 32, 84, 1, 1), (6, 60, 57, 16, 100, 3, 1)]


@pytest.mark.parametrize("off", OFFSETS)
@pytest.mark.parametrize("case", CONV)
def test_int8(ctx, case, off):
    n, h, w, ic, oc, k, stride = case
    rng = np.random.default_rng(ic + oc)
    x, wt = rng.integers(-128, 128, (n, h, w, ic)).astype(np.int8), rng.integers(-128, 128, (oc, k, k, ic)).astype(np.int8)
    bias = rng.integers(-9999, 9999, oc).astype(np.int32)
    d, shape = _conv_desc(ctx, capi.INT8, capi.INT32, x, oc, k, stride)
    out = ctx.empty(shape, capi.INT32)
    ctx.conv2d(d, _put(ctx, x, off[0]), _put(ctx, wt, off[1]), ctx.upload(bias), -11, 0, out)
    assert ctx.sync() == capi.VALID and ctx.last_kernel == "conv2d_taps_i8"
    assert np.array_equal(out.numpy(), oracle.conv2d("i8", x, wt, bias, (k // 2,) * 4, (stride, stride), (1, 1), in_zp=-11, w_zp=0))


@pytest.mark.parametrize("dtype", [capi.FP16, capi.BF16])
@pytest.mark.parametrize("off", OFFSETS)
@pytest.mark.parametrize("case", [(n, h, w, ic // 2, oc, k, s) for n, h, w, ic, oc, k, s in CONV])
def test_16_bit_floats(ctx, case, off, dtype):
    n, h, w, ic, oc, k, stride = case
    rng = np.random.default_rng(ic + oc)
    # (whole quarters: products and sums are exact in fp32)
    x, wt, bias = (rng.integers(-8, 9, s).astype(np.float32) / 4 for s in ((n, h, w, ic), (oc, k, k, ic), (oc,)))
    ax, aw, ab = (v.astype(np.float16) if dtype == capi.FP16 else (v.view(np.uint32) >> 16).astype(np.uint16) for v in (x, wt, bias))
    d, shape = _conv_desc(ctx, dtype, dtype, x, oc, k, stride)
    out = ctx.empty(shape, dtype)
    ctx.conv2d(d, _put(ctx, ax, 2 * off[0]), _put(ctx, aw, 2 * off[1]), ctx.upload(ab, dtype), 0, 0, out)
    assert ctx.sync() == capi.VALID and ctx.last_kernel == ("conv2d_taps_f16" if dtype == capi.FP16 else "conv2d_taps_bf16")
    got = out.numpy().astype(np.float64) if dtype == capi.FP16 else (out.numpy().astype(np.uint32) << 16).view(np.float32).astype(np.float64)
    want = oracle.conv2d("f64", *(v.astype(np.float64) for v in (x, wt, bias)), (k // 2,) * 4, (stride, stride), (1, 1))
    assert np.all(np.abs(got - want) <= (2.0 ** -11 if dtype == capi.FP16 else 2.0 ** -8) * np.abs(want))


@pytest.mark.parametrize("off", OFFSETS)
@pytest.mark.parametrize("case", [(1, 10, 25, 16, 33, 1, 1), (3, 33, 31, 16, 15, 3, 1), (4, 60, 60, 16, 64, 3, 1), (5, 90, 91, 32, 21, 1, 1)])
def test_int16(ctx, case, off):
    n, h, w, ic, oc, k, stride = case
    rng = np.random.default_rng(ic + oc)
    x, wt = rng.integers(-32768, 32768, (n, h, w, ic)).astype(np.int16), rng.integers(-128, 128, (oc, k, k, ic)).astype(np.int8)
    bias = rng.integers(-(1 << 40), 1 << 40, oc).astype(np.int64)
    d, shape = _conv_desc(ctx, capi.INT16, capi.INT48, x, oc, k, stride)
    out = ctx.empty(shape, capi.INT48)
    ctx.conv2d(d, _put(ctx, x, 2 * off[0]), _put(ctx, wt, off[1]), ctx.upload(bias), 0, 0, out)
    assert ctx.sync() == capi.VALID and ctx.last_kernel == "conv2d_mfma_i16_i48"
    assert np.array_equal(out.numpy(), oracle.conv2d("i16", x, wt, bias, (k // 2,) * 4, (stride, stride), (1, 1)))


@pytest.mark.parametrize("off", OFFSETS)
@pytest.mark.parametrize("case", [(1, 7, 9, 16, 17, 2), (2, 9, 11, 48, 16, 3), (3, 13, 12, 32, 128, 4), (2, 60, 61, 16, 12, 3)])
def test_transpose_conv2d(ctx, case, off):
    n, h, w, ic, oc, k = case
    rng = np.random.default_rng(ic + oc)
    x, wt = rng.integers(-128, 128, (n, h, w, ic)).astype(np.int8), rng.integers(-128, 128, (oc, k, k, ic)).astype(np.int8)
    bias = rng.integers(-9999, 9999, oc).astype(np.int32)
    d = capi.TconvDesc()
    d.in_dtype, d.out_dtype = capi.INT8, capi.INT32
    d.N, d.IH, d.IW, d.IC, d.OC, d.KH, d.KW, d.OH, d.OW = n, h, w, ic, oc, k, k, (h - 1) * 2 + k, (w - 1) * 2 + k
    d.out_pad[:], d.stride[:], d.bias_len = [0] * 4, [2, 2], oc
    out = ctx.empty((n, d.OH, d.OW, oc), capi.INT32)
    ctx.transpose_conv2d(d, _put(ctx, x, off[0]), _put(ctx, wt, off[1]), ctx.upload(bias), -7, 0, out)
    assert ctx.sync() == capi.VALID and ctx.last_kernel == "transpose_conv2d_taps_i8"
    assert np.array_equal(out.numpy(), oracle.transpose_conv2d("i8", x, wt, bias, (0, 0, 0, 0), (2, 2), -7, 0))


@pytest.mark.parametrize("off", OFFSETS)
@pytest.mark.parametrize("case", [(2, 10, 9, 16, 5, 1), (1, 12, 12, 8, 5, 2), (8, 60, 60, 44, 3, 1), (3, 79, 63, 28, 3, 2)])
def test_depthwise(ctx, case, off):
    n, h, w, c, k, stride = case
    rng = np.random.default_rng(c)
    x, wt = rng.integers(-128, 128, (n, h, w, c)).astype(np.int8), rng.integers(-128, 128, (k, k, c, 1)).astype(np.int8)
    bias = rng.integers(-9999, 9999, c).astype(np.int32)
    pad = (k // 2, k // 2 - (h + 2 * (k // 2) - k) % stride, k // 2, k // 2 - (w + 2 * (k // 2) - k) % stride)
    oh, ow = oracle.conv_out_hw(h, w, k, k, pad, (stride, stride), (1, 1))
    d = ctx.conv_desc(capi.INT8, capi.INT32, x.shape, c, k, k, (oh, ow), pad, (stride, stride), (1, 1), c)
    out = ctx.empty((n, oh, ow, c), capi.INT32)
    ctx.depthwise_conv2d(d, _put(ctx, x, off[0]), _put(ctx, wt, off[1]), ctx.upload(bias), 9, 0, out)
    assert ctx.sync() == capi.VALID and ctx.last_kernel == "depthwise_rows_i8"
    assert np.array_equal(out.numpy(), oracle.depthwise_conv2d("i8", x, wt, bias, pad, (stride, stride), in_zp=9, w_zp=0))
