"""MATMUL and CONV2D whose rows begin between words, read from the word before: every split of K, pieces at the end of a row, of K and of the
tensor.  Values are small whole numbers, so that sums in any order are exact."""
import numpy as np
import pytest

import oracle
from reference_model_amd import Context, capi

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = Context(0)
    yield c
    c.close()


@pytest.mark.parametrize("shape", [  # n, h, c, w
    (1, 33, 33, 65), (2, 5, 95, 63), (3, 31, 127, 67), (1, 1, 191, 2), (7, 40, 203, 33), (1, 64, 333, 129), (2, 14, 2529, 160), (1, 13, 1601, 37),
    (300, 33, 65, 67), (260, 31, 63, 127), (600, 40, 33, 70)])    # a wave to a tile
@pytest.mark.parametrize("dtype, offset", [("int8", 0), ("int8", 1), ("int8", 2), ("int8", 3), ("fp16", 0), ("fp16", 1), ("bf16", 1)])
def test_rows_between_words(ctx, shape, dtype, offset):
    n, h, c, w = shape
    rng = np.random.default_rng(c * w)
    a, b = rng.integers(-8, 9, n * h * c).astype(np.int8), rng.integers(-8, 9, n * c * w).astype(np.int8)
    store = {"int8": lambda v: v, "fp16": lambda v: v.astype(np.float16), "bf16": lambda v: (v.astype(np.float32).view(np.uint32) >> 16).astype(np.uint16)}[dtype]
    code, eb = {"int8": (capi.INT8, 1), "fp16": (capi.FP16, 2), "bf16": (capi.BF16, 2)}[dtype]
    za, zb = (-3, 5) if dtype == "int8" else (0, 0)
    bad = np.full(offset, 127 if dtype == "int8" else np.nan if dtype == "fp16" else 0x7fc0, store(a[:1]).dtype)    # what lies before the operands counts for nothing
    ta, tb = (ctx.upload(np.concatenate([bad, store(v)]), code) for v in (a, b))
    out = ctx.empty((n, h, w), capi.INT32 if dtype == "int8" else capi.FP32)
    ctx.matmul(code, n, h, c, w, ta.ptr + offset * eb, tb.ptr + offset * eb, za, zb, out)
    assert ctx.sync() == capi.VALID and "ragged" in ctx.last_kernel
    want = np.matmul(a.reshape(n, h, c).astype(np.float64) - za, b.reshape(n, c, w).astype(np.float64) - zb)
    assert np.array_equal(out.numpy().astype(np.float64), want)
    for t in (ta, tb, out):
        t.free()


@pytest.mark.parametrize("shape", [  # n, h, w, ic, oc, k, stride
    (1, 5, 7, 33, 17, 1, 1), (2, 9, 8, 35, 40, 3, 1), (1, 8, 9, 49, 8, 3, 2), (1, 6, 5, 101, 33, 2, 1), (1, 10, 11, 163, 24, 3, 1), (2, 4, 4, 331, 9, 5, 1),
    (9, 40, 40, 57, 12, 3, 1), (40, 20, 20, 163, 20, 1, 1), (30, 21, 20, 37, 70, 3, 1), (24, 30, 30, 41, 100, 1, 1)])    # weights resident: several tiles a wave
@pytest.mark.parametrize("dtype, offset", [("int8", 0), ("int8", 1), ("int8", 2), ("fp16", 0), ("fp16", 1), ("bf16", 1)])
def test_channel_vectors_between_words(ctx, shape, dtype, offset):
    n, h, w, ic, oc, k, s = shape
    rng = np.random.default_rng(ic * oc)
    x, wt, bias = rng.integers(-4, 5, (n, h, w, ic)), rng.integers(-2, 3, (oc, k, k, ic)), rng.integers(-9, 10, oc)
    store = {"int8": lambda v: v.astype(np.int8), "fp16": lambda v: v.astype(np.float16), "bf16": lambda v: (v.astype(np.float32).view(np.uint32) >> 16).astype(np.uint16)}[dtype]
    code, eb = {"int8": (capi.INT8, 1), "fp16": (capi.FP16, 2), "bf16": (capi.BF16, 2)}[dtype]
    p = k // 2
    pad = (p, p - (h + 2 * p - k) % s, p, p - (w + 2 * p - k) % s)
    oh, ow = oracle.conv_out_hw(h, w, k, k, pad, (s, s), (1, 1))
    bad = np.full(offset, 127 if dtype == "int8" else np.nan if dtype == "fp16" else 0x7fc0, store(np.zeros(1)).dtype)    # counts for nothing, before and behind
    tx, tw = (ctx.upload(np.concatenate([bad, store(v).ravel(), bad]), code) for v in (x, wt))
    tb = ctx.upload(bias.astype(np.int32) if dtype == "int8" else store(bias), capi.INT32 if dtype == "int8" else code)
    out = ctx.empty((n, oh, ow, oc), capi.INT32 if dtype == "int8" else code)
    d = ctx.conv_desc(code, capi.INT32 if dtype == "int8" else code, (n, h, w, ic), oc, k, k, (oh, ow), pad, (s, s), (1, 1), oc)
    za = -11 if dtype == "int8" else 0
    ctx.conv2d(d, tx.ptr + offset * eb, tw.ptr + offset * eb, tb, za, 0, out)
    assert ctx.sync() == capi.VALID
    want = oracle.conv2d("f64", x.astype(np.float64) - za, wt.astype(np.float64), bias.astype(np.float64), pad, (s, s), (1, 1))
    got = out.numpy()
    if dtype == "bf16":
        got = (got.astype(np.uint32) << 16).view(np.float32)
    ulp = {"int8": 0.0, "fp16": 2.0 ** -11, "bf16": 2.0 ** -8}[dtype]    # the sum is exact: one rounding of the result
    assert np.all(np.abs(got.astype(np.float64) - want) <= ulp * np.abs(want))
    for t in (tx, tw, tb, out):
        t.free()


EVERY, FLOATS = ("int8", "fp16", "bf16"), ("fp16", "bf16")
ON_COPIES = {    # 36 steps and more with taps; more than 18 on many tiles; many tiles and channels
    (1, 10, 11, 163, 24, 3, 1): EVERY, (2, 4, 4, 331, 9, 5, 1): EVERY, (9, 40, 40, 57, 12, 3, 1): FLOATS, (30, 21, 20, 37, 40, 3, 1): FLOATS,
    (5, 32, 33, 939, 200, 1, 1): FLOATS}    # (of many channels: to the GEMM kernel)


@pytest.mark.parametrize("shape", [  # n, h, w, ic, oc, k, stride
    (1, 5, 7, 33, 17, 1, 1), (2, 9, 8, 35, 40, 3, 1), (1, 8, 9, 49, 8, 3, 2), (1, 6, 5, 101, 33, 2, 1), (1, 10, 11, 163, 24, 3, 1), (2, 4, 4, 331, 9, 5, 1), (1, 10, 11, 467, 24, 1, 1), (2, 4, 4, 1331, 9, 1, 1),
    (9, 40, 40, 57, 12, 3, 1), (40, 20, 20, 163, 20, 1, 1), (30, 21, 20, 37, 40, 3, 1), (12, 40, 40, 29, 12, 3, 1), (24, 30, 30, 41, 100, 1, 1),    # weights resident: several tiles a wave
    (33, 32, 32, 761, 24, 1, 1), (33, 32, 32, 829, 18, 1, 1), (33, 32, 32, 930, 9, 1, 1), (5, 32, 33, 939, 200, 1, 1)])    # int8: K split, two tiles a workgroup on shares of six (kept in registers), seven and eight steps; too many channels for that
@pytest.mark.parametrize("dtype, offset", [("int8", 0), ("int8", 1), ("int8", 2), ("fp16", 0), ("fp16", 1), ("bf16", 1)])
def test_channel_vectors_between_words_as_they_lie_or_on_copies(shape, dtype, offset):
    ctx = Context(0)    # (one that has no scratch yet: whether the layer ran on copies)
    try:
        test_channel_vectors_between_words(ctx, shape, dtype, offset)
        copied = dtype in ON_COPIES.get(shape, ())
        assert (ctx.workspace_bytes() != (0, 0)) == copied and (copied or "taps" in ctx.last_kernel)
    finally:
        ctx.close()
