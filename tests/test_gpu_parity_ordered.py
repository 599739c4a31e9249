"""The ordered tiles (fp32 CONV2D / MATMUL and the fp64 passes): bit for bit the oracle's loop nest, at the edges of the tiles
and stages, in every way the first operand is read, and where a weight is infinite under a tap outside the image."""
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


# n, ih, iw, ic, oc, k, pad, stride; reductions of whole units of eight channels from 224 (the fp32 operator: 400) on run on operands staged through LDS
STAGED = [
    (1, 8, 8, 32, 64, 3, 1, 1),
    (1, 5, 13, 64, 65, 3, 1, 1),
    (2, 9, 7, 96, 31, 3, 1, 2),
]
CONVS = STAGED + [
    (1, 9, 9, 32, 64, 2, 0, 1),      # one whole tile, stages inside a tap
    (1, 6, 14, 32, 65, 2, 0, 1),     # one row and one column past a tile
    (2, 9, 7, 32, 31, 2, 1, 2),      # narrow channels: 64 x 32 tiles
    (1, 5, 5, 32, 200, 2, 0, 1),     # few pixels: 32 x 64 tiles
    (1, 9, 9, 20, 70, 3, 1, 1),      # groups of four, stages across taps
    (2, 7, 9, 5, 66, 3, 1, 1),       # single elements
    (1, 9, 9, 16, 72, 1, 0, 1),      # a short reduction
    (1, 63, 64, 32, 256, 2, 1, 1),   # 65 x 4 tiles: a whole round and four cut into quarters, the last row ragged
    (1, 63, 64, 28, 200, 2, 1, 1),   # the same across taps, the last column ragged
    (1, 63, 64, 12, 200, 2, 1, 1),   # a short reduction: whole tiles
]


@pytest.mark.parametrize("case", CONVS)
@pytest.mark.parametrize("infinite", [False, True])
def test_conv2d_in_the_references_order(ctx, case, infinite):
    n, ih, iw, ic, oc, k, p, s = case
    tiles = "_ordered" if case == CONVS[-1] else "_ordered_staged" if case in STAGED else "_ordered_tail"
    op_tiles = "_ordered_tail" if case == STAGED[0] else tiles
    rng = np.random.default_rng(ic * oc)
    x = rng.normal(0, 1, (n, ih, iw, ic)).astype(np.float32)
    w = rng.normal(0, 0.3, (oc, k, k, ic)).astype(np.float32)
    b = rng.normal(0, 1, oc).astype(np.float32)
    if infinite:
        w[oc // 2, 0, 0, 1] = np.inf
    pad = (p, p, p, p)
    if s == 2:
        pad = (p, p - (ih + 2 * p - k) % 2, p, p - (iw + 2 * p - k) % 2)
    oh, ow = oracle.conv_out_hw(ih, iw, k, k, pad, (s, s), (1, 1))
    with np.errstate(invalid="ignore"):
        want = oracle.conv2d("f32", x, w, b, pad, (s, s), (1, 1))
        got, st = gpu_ops.conv2d(ctx, x, w, b, pad, (s, s), (1, 1), dtype=capi.FP32)
        assert st == capi.VALID and np.array_equal(got, want, equal_nan=True) and ctx.last_kernel == "conv2d" + op_tiles + "_f32"
        d = ctx.conv_desc(capi.FP32, capi.FP32, x.shape, oc, k, k, (oh, ow), pad, (s, s), (1, 1), oc)
        dev = [ctx.upload(v) for v in (x, w, b)]
        for bounds in (False,) if infinite else (False, True):    # (the oracle's bounds pass multiplies the padding out: NaN)
            out = ctx.empty((n, oh, ow, oc), capi.F64)
            ctx.conv2d_precise(d, *dev, bounds, out)
            assert ctx.sync() == capi.VALID and ctx.last_kernel == ("conv_bounds" if bounds else "conv_precise") + tiles + "_f64"
            want = oracle.conv2d("f64", *(v.astype(np.float64) for v in (x, w, b)), pad, (s, s), (1, 1), abs_mode=bounds)
            assert np.array_equal(out.numpy(), want, equal_nan=True)


@pytest.mark.parametrize("shape", [(1, 64, 32, 64), (2, 65, 33, 63), (3, 5, 17, 130), (1, 130, 100, 7), (2, 1, 3, 1), (1, 70, 96, 66),
                                   # a whole round of tiles, and one with quarters behind; short stages, 64 x 32, 32 x 64; batches
                                   (1, 1024, 50, 1000), (1, 4097, 64, 250), (1, 4097, 35, 250), (1, 16600, 50, 20), (1, 20, 50, 16600),
                                   (1, 4097, 40, 250), (70, 100, 33, 70), (48, 100, 33, 70)])
def test_matmul_in_the_references_order(ctx, shape):
    n, h, c, w = shape
    # more than 192 tiles, and none or none that could be cut left over by whole rounds
    tiles = "_ordered" if shape in ((1, 1024, 50, 1000), (1, 4097, 35, 250), (1, 16600, 50, 20), (1, 20, 50, 16600), (1, 4097, 40, 250),
                                    (70, 100, 33, 70)) else "_ordered_tail"
    rng = np.random.default_rng(h * c)
    a, b = rng.normal(0, 1, (n, h, c)).astype(np.float32), rng.normal(0, 1, (n, c, w)).astype(np.float32)
    got, st = gpu_ops.matmul(ctx, a, b, dtype=capi.FP32)
    assert st == capi.VALID and np.array_equal(got, oracle.matmul("f32", a, b)) and ctx.last_kernel == "matmul" + tiles + "_f32"
    da, db = ctx.upload(a), ctx.upload(b)
    for bounds in (False, True):
        out = ctx.empty((n, h, w), capi.F64)
        ctx.matmul_precise(capi.FP32, n, h, c, w, da, db, bounds, out)
        assert ctx.sync() == capi.VALID and ctx.last_kernel == ("matmul_bounds" if bounds else "matmul_precise") + tiles + "_f64"
        assert np.array_equal(out.numpy(), oracle.matmul("f64", a.astype(np.float64), b.astype(np.float64), abs_mode=bounds))
