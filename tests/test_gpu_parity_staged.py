"""The ordered sums on units of eight channels staged through LDS (fp64 passes, fp32 operator on few tiles): bit for bit the oracle's loop
nest at the edges of tiles, units, stages and taps, and where a weight is infinite under a tap outside the image."""
import time

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


CASES = [  # n, ih, iw, ic, oc, kh, kw, pads, strides, dilations
    (1, 4, 4, 104, 16, 1, 1, (0, 0, 0, 0), (1, 1), (1, 1)),        # thirteen units, no padding, half a tile of channels
    (2, 7, 5, 16, 33, 3, 3, (1, 1, 1, 1), (1, 1), (1, 1)),         # two units a tap: lanes of a stage under different taps
    (1, 6, 9, 8, 17, 5, 4, (2, 2, 1, 2), (1, 2), (1, 1)),          # one unit a tap, uneven padding
    (3, 5, 9, 40, 70, 3, 3, (2, 2, 2, 2), (1, 1), (2, 2)),         # dilated: K 360, a last stage of one unit
    (1, 18, 11, 56, 20, 3, 3, (1, 0, 0, 1), (2, 1), (1, 2)),       # K 504
    (1, 9, 8, 64, 65, 3, 3, (1, 1, 1, 1), (1, 1), (1, 1)),         # whole stages, one column past a tile
    (1, 66, 65, 32, 250, 3, 3, (1, 1, 1, 1), (1, 1), (1, 1)),      # a whole round of tiles and quarters, whole stages
    (1, 66, 65, 24, 250, 3, 3, (1, 1, 1, 1), (1, 1), (1, 1)),      # the same across taps
    (1, 2, 3, 128, 33, 3, 3, (1, 1, 1, 1), (1, 1), (1, 1)),        # six pixels
    (1, 1, 1, 512, 5, 1, 1, (0, 0, 0, 0), (1, 1), (1, 1)),         # one
]


@pytest.mark.parametrize("case", CASES)
@pytest.mark.parametrize("dtype", ["fp32", "fp16", "bf16"])
@pytest.mark.parametrize("infinite", [False, True])
def test_conv2d_staged(ctx, case, dtype, infinite):
    n, ih, iw, ic, oc, kh, kw, pad, stride, dil = case
    rng = np.random.default_rng(ic * oc)
    x, w, b = rng.normal(0, 1, (n, ih, iw, ic)), rng.normal(0, 0.3, (oc, kh, kw, ic)), rng.normal(0, 1, oc if ic % 3 else 1)
    if infinite:
        w[oc // 2, 0, 0, 1] = np.inf
    if dtype == "bf16":    # the bits of values that bf16 holds
        bits = [(v.astype(np.float32).view(np.uint32) >> 16).astype(np.uint16) for v in (x, w, b)]
        x, w, b = ((v.astype(np.uint32) << 16).view(np.float32) for v in bits)
    else:
        bits = x, w, b = tuple(v.astype(np.float32 if dtype == "fp32" else np.float16) for v in (x, w, b))
    code = {"fp32": capi.FP32, "fp16": capi.FP16, "bf16": capi.BF16}[dtype]
    oh, ow = oracle.conv_out_hw(ih, iw, kh, kw, pad, stride, dil)
    bias = np.broadcast_to(b, oc)
    staged_op = ic * kh * kw >= 400 and n * oh * ow * oc <= 192 * 64 * 64    # (the fp32 operator stages long reductions on few tiles)
    d = ctx.conv_desc(code, code, (n, ih, iw, ic), oc, kh, kw, (oh, ow), pad, stride, dil, len(b))
    with np.errstate(invalid="ignore"):
        if dtype == "fp32":
            got, st = gpu_ops.conv2d(ctx, x, w, b, pad, stride, dil, dtype=capi.FP32)
            assert st == capi.VALID and (ctx.last_kernel == "conv2d_ordered_staged_f32") == staged_op and np.array_equal(got, oracle.conv2d("f32", x, w, bias, pad, stride, dil), equal_nan=True)
        dev = [ctx.upload(np.ascontiguousarray(v), code) for v in bits]    # (behind gpu_ops, which frees the context's tensors)
        for bounds in (False, True):    # (the bounds pass multiplies the padding out: an infinite weight there makes NaN)
            out = ctx.empty((n, oh, ow, oc), capi.F64)
            ctx.conv2d_precise(d, *dev, bounds, out)
            assert ctx.sync() == capi.VALID and ctx.last_kernel == ("conv_bounds" if bounds else "conv_precise") + "_ordered_staged_f64"
            want = oracle.conv2d("f64", *(v.astype(np.float64) for v in (x, w, bias)), pad, stride, dil, abs_mode=bounds)
            assert np.array_equal(out.numpy(), want, equal_nan=True)


@pytest.mark.parametrize("dtype, precise", [("fp32", False), ("fp32", True), ("bf16", True)])
def test_a_nan_image_costs_no_sums(ctx, dtype, precise):
    """A result that is NaN through its window costs a look at the weights; summed again one product after the other it took 25 to 37 times as long."""
    rng = np.random.default_rng(1)
    n, h, w, ic, oc = 4, 14, 14, 256, 64
    store = {"fp32": lambda v: v.astype(np.float32), "bf16": lambda v: (v.astype(np.float32).view(np.uint32) >> 16).astype(np.uint16)}[dtype]
    code = {"fp32": capi.FP32, "bf16": capi.BF16}[dtype]
    wt, b = ctx.upload(store(rng.normal(0, 0.1, (oc, 3, 3, ic))), code), ctx.upload(store(np.zeros(oc)), code)
    d = ctx.conv_desc(code, code, (n, h, w, ic), oc, 3, 3, (h, w), (1, 1, 1, 1), (1, 1), (1, 1), oc)
    out = ctx.empty((n, h, w, oc), capi.F64 if precise else code)

    def seconds(x):
        call = (lambda: ctx.conv2d_precise(d, x, wt, b, False, out)) if precise else (lambda: ctx.conv2d(d, x, wt, b, 0, 0, out))
        call(), ctx.sync()
        start = time.perf_counter()
        for _ in range(10):
            call()
        assert ctx.sync() == capi.VALID and "ordered_staged" in ctx.last_kernel
        return time.perf_counter() - start
    finite = seconds(ctx.upload(store(rng.normal(0, 1, (n, h, w, ic))), code))
    nan = seconds(ctx.upload(store(np.full((n, h, w, ic), np.nan)), code))
    print("us a call, finite / NaN:", finite / 10e-6, nan / 10e-6)
    assert np.isnan(out.numpy()).all() and nan < 4 * finite
