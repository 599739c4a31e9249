"""The ordered sums on copies of the operands (fp32 CONV2D and its fp64 passes): bit for bit the oracle's loop nest, at the edges of tiles,
granules and stages, and where a weight is infinite under a tap outside the image."""
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


CASES = [  # n, ih, iw, ic, oc, kh, kw, pads, strides, dilations, fp32 sums on copies too
    (1, 5, 6, 50, 33, 3, 3, (1, 1, 1, 1), (1, 1), (1, 1), True),       # 450: single elements, odd granules, one column past a tile
    (2, 4, 5, 45, 7, 3, 3, (1, 0, 1, 0), (1, 1), (1, 1), True),        # few channels
    (1, 9, 9, 26, 66, 3, 3, (1, 1, 1, 1), (2, 2), (1, 1), False),      # 234
    (1, 7, 8, 65, 64, 2, 4, (2, 2, 1, 3), (1, 2), (2, 1), True),       # dilated, strided, uneven padding
    (1, 6, 4, 116, 40, 3, 3, (1, 1, 1, 1), (1, 1), (1, 1), True),      # 1044, whole groups of four
    (1, 6, 5, 128, 65, 3, 3, (0, 0, 0, 0), (1, 1), (1, 1), False),     # 1152, whole stages, no padding: copies for the bounds pass of the largest magnitude
    (1, 7, 6, 60, 65, 4, 4, (0, 0, 0, 0), (1, 1), (1, 1), False),      # 960, whole stages
    (1, 2, 3, 51, 5, 2, 2, (0, 0, 0, 0), (1, 1), (1, 1), False),       # two results in a row of 204
    (1, 114, 113, 59, 65, 2, 2, (1, 0, 0, 1), (1, 1), (1, 1), False),  # a whole round of tiles and quarters
]


@pytest.mark.parametrize("case", CASES)
@pytest.mark.parametrize("infinite", [False, True])
def test_conv2d_on_copies(ctx, case, infinite):
    n, ih, iw, ic, oc, kh, kw, pad, stride, dil, f32 = case
    rng = np.random.default_rng(ic * oc)
    x = rng.normal(0, 1, (n, ih, iw, ic)).astype(np.float32)
    w = rng.normal(0, 0.3, (oc, kh, kw, ic)).astype(np.float32)
    b = rng.normal(0, 1, oc if ic % 2 else 1).astype(np.float32)
    if infinite:
        w[oc // 2, 0, 0, 1] = np.inf
    oh, ow = oracle.conv_out_hw(ih, iw, kh, kw, pad, stride, dil)
    bias = np.broadcast_to(b, oc)
    with np.errstate(invalid="ignore"):
        if f32:
            got, st = gpu_ops.conv2d(ctx, x, w, b, pad, stride, dil, dtype=capi.FP32)
            assert st == capi.VALID and ctx.last_kernel == "conv2d_copied_f32"
            assert np.array_equal(got, oracle.conv2d("f32", x, w, bias, pad, stride, dil), equal_nan=True)
        d = ctx.conv_desc(capi.FP32, capi.FP32, x.shape, oc, kh, kw, (oh, ow), pad, stride, dil, len(b))
        dev = [ctx.upload(v) for v in (x, w, b)]
        for bounds in (False, True):    # (the bounds pass multiplies the padding out: an infinite weight there makes NaN)
            for local in (True, False) if bounds else (True,):
                out = ctx.empty((n, oh, ow, oc), capi.F64)
                ctx.conv2d_precise(d, *dev, bounds, out, local_bound=local)
                kind = "_ordered_staged_f64" if ic % 8 == 0 and local else "_copied_f64"    # (units of eight channels are staged as they lie)
                assert ctx.sync() == capi.VALID and ctx.last_kernel == ("conv_bounds" if bounds else "conv_precise") + kind
                xs = x.astype(np.float64) if local else np.full(x.shape, np.abs(x).max(), np.float64)
                want = oracle.conv2d("f64", xs, w.astype(np.float64), bias.astype(np.float64), pad, stride, dil, abs_mode=bounds)
                assert np.array_equal(out.numpy(), want, equal_nan=True)


@pytest.mark.parametrize("dtype", ["fp16", "bf16"])
def test_precise_pass_of_sixteen_bit_operands(ctx, dtype):
    """An image of infinities and NaN: only products of its own elements may see them."""
    rng = np.random.default_rng(5)
    ih, iw, ic, oc = 6, 7, 27, 35
    x, w, b = (rng.integers(-8, 9, s).astype(np.float32) / 4 for s in ((1, ih, iw, ic), (oc, 3, 3, ic), (oc,)))
    x[0, 2, 3, ic - 1], x[0, 5, 6, 0] = np.inf, np.nan
    code = capi.FP16 if dtype == "fp16" else capi.BF16
    narrow = (lambda v: v.astype(np.float16)) if dtype == "fp16" else (lambda v: (v.view(np.uint32) >> 16).astype(np.uint16))    # (exact)
    d = ctx.conv_desc(code, code, x.shape, oc, 3, 3, (ih, iw), (1, 1, 1, 1), (1, 1), (1, 1), oc)
    dev = [ctx.upload(narrow(v), code) for v in (x, w, b)]
    out = ctx.empty((1, ih, iw, oc), capi.F64)
    ctx.conv2d_precise(d, *dev, False, out)
    assert ctx.sync() == capi.VALID and ctx.last_kernel == "conv_precise_copied_f64"
    with np.errstate(invalid="ignore"):
        want = oracle.conv2d("f64", *(v.astype(np.float64) for v in (x, w, b)), (1, 1, 1, 1), (1, 1), (1, 1))
    assert np.array_equal(out.numpy(), want, equal_nan=True)


@pytest.mark.parametrize("shape, kernel", [
    ((2, 9, 8, 12, 20), "conv_bounds_ordered"),       # read as they lie
    ((2, 9, 8, 64, 40), "conv_bounds_ordered"),       # channels of whole stages
    ((1, 2, 65536, 1, 2), "conv_bounds_f64")])        # too wide for the tiles: one result a lane
@pytest.mark.parametrize("local", [True, False])
def test_bounds_pass_multiplies_the_padding_out(ctx, shape, kernel, local):
    """an infinite weight under a tap outside the image: NaN in the bounds pass, nothing in the others"""
    n, h, w, ic, oc = shape
    rng = np.random.default_rng(ic)
    x, wt, b = rng.normal(0, 1, (n, h, w, ic)).astype(np.float32), rng.normal(0, 0.3, (oc, 3, 3, ic)).astype(np.float32), rng.normal(0, 1, oc).astype(np.float32)
    wt[oc // 2, 0, 0, 0], wt[0, 2, 1, ic - 1] = -np.inf, np.nan
    d = ctx.conv_desc(capi.FP32, capi.FP32, x.shape, oc, 3, 3, (h, w), (1, 1, 1, 1), (1, 1), (1, 1), oc)
    dev = [ctx.upload(v) for v in (x, wt, b)]
    for bounds in (False, True):
        out = ctx.empty((n, h, w, oc), capi.F64)
        ctx.conv2d_precise(d, *dev, bounds, out, local_bound=local)
        assert ctx.sync() == capi.VALID and ctx.last_kernel.startswith(kernel if bounds else kernel.replace("bounds", "precise"))
        xs = np.full(x.shape, np.abs(x).max()) if bounds and not local else x
        with np.errstate(invalid="ignore"):
            want = oracle.conv2d("f64", *(v.astype(np.float64) for v in (xs, wt, b)), (1, 1, 1, 1), (1, 1), (1, 1), abs_mode=bounds)
        assert np.array_equal(out.numpy(), want, equal_nan=True)
        assert np.isnan(want).any() and np.isinf(want).any()


@pytest.mark.parametrize("case, f64, copied", [  # n, ih, iw, ic, oc, k
    ((10, 61, 64, 21, 30, 5), False, False),     # 610 tiles of few channels: either operand read for half a tile of results
    ((10, 57, 64, 21, 30, 5), False, True),      # 570
    ((10, 64, 64, 112, 8, 3), True, False),      # 640
    ((2, 52, 41, 53, 96, 3), False, False),      # 134 tiles in quarters, K 477
    ((2, 52, 41, 63, 96, 3), False, True),       # K 567
    ((1, 20, 20, 6, 40, 11), False, False),      # few channels: the granules would be filled up with zeros
    ((1, 20, 20, 4, 40, 17), False, False),
    ((1, 20, 20, 28, 40, 7), False, True),
    ((1, 20, 20, 2, 40, 13), True, False),
    ((1, 20, 20, 4, 40, 17), True, False),
    ((1, 20, 20, 5, 40, 13), True, True)])
def test_copies_where_they_lead(case, f64, copied):
    n, h, w, ic, oc, k = case
    c = Context(0)
    try:
        d = c.conv_desc(capi.FP32, capi.FP32, (n, h, w, ic), oc, k, k, (h, w), (k // 2,) * 4, (1, 1), (1, 1), oc)
        dev = [c.upload(np.zeros(s, np.float32)) for s in ((n, h, w, ic), (oc, k, k, ic), (oc,))]
        out = c.empty((n, h, w, oc), capi.F64 if f64 else capi.FP32)
        c.conv2d_precise(d, *dev, False, out) if f64 else c.conv2d(d, *dev, 0, 0, out)
        assert c.sync() == capi.VALID and ("copied" in c.last_kernel) == copied and not out.numpy().any()
    finally:
        c.close()
