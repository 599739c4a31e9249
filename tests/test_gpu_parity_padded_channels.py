"""CONV2D whose channel vectors are no whole steps of the matrix instruction: copies padded with zeros, then the kernels for whole
vectors.  Bit for bit against the oracle for int8; fp16 and bf16 against fp64 within fp32 accumulation and one rounding of the result."""
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


CASES = [  # n, h, w, ic, oc, k, pad, stride
    (1, 7, 9, 17, 24, 3, 1, 1),       # one byte past a piece
    (2, 9, 7, 31, 8, 3, 1, 1),        # one short of a step
    (1, 8, 8, 33, 13, 1, 0, 1),
    (3, 11, 5, 131, 40, 3, 1, 2),
    (1, 6, 6, 207, 64, 2, 0, 1),
    (2, 13, 13, 72, 72, 3, 1, 1),     # whole words, the K-split kernel
    (2, 12, 12, 80, 80, 3, 1, 1),     # the slab kernel
    (1, 10, 10, 245, 16, 3, 1, 1),    # padded to 256: both operands in LDS
]


@pytest.mark.parametrize("case", CASES)
@pytest.mark.parametrize("fused", [False, True])
def test_int8(ctx, case, fused):
    n, h, w, ic, oc, k, p, s = case
    rng = np.random.default_rng(ic)
    x = rng.integers(-128, 128, (n, h, w, ic)).astype(np.int8)
    wt = rng.integers(-128, 128, (oc, k, k, ic)).astype(np.int8)
    bias = rng.integers(-9999, 9999, oc).astype(np.int32)
    pad = (p, p - (h + 2 * p - k) % s, p, p - (w + 2 * p - k) % s)
    want = oracle.conv2d("i8", x, wt, bias, pad, (s, s), (1, 1), in_zp=-11, w_zp=0)
    if not fused:
        got, st = gpu_ops.conv2d(ctx, x, wt, bias, pad, (s, s), in_zp=-11, w_zp=0)
        assert st == capi.VALID and np.array_equal(got, want)
        return
    mult, shift = rng.integers(1 << 30, 1 << 31, oc).astype(np.int32), rng.integers(38, 43, oc).astype(np.int8)
    want, wst = oracle.rescale(want, mult, shift, out_zp=3)
    got, st = gpu_ops.conv2d(ctx, x, wt, bias, pad, (s, s), in_zp=-11, w_zp=0, rescale=dict(mult=mult, shift=shift, out_zp=3))
    assert st == wst and np.array_equal(got, want) and len(np.unique(got)) > 20


@pytest.mark.parametrize("case", CASES + [(1, 9, 9, 9, 16, 3, 1, 1), (1, 9, 9, 100, 40, 3, 1, 1), (2, 12, 12, 40, 64, 3, 1, 1)])
@pytest.mark.parametrize("dtype", [capi.FP16, capi.BF16])
def test_16_bit_floats(ctx, case, dtype):
    n, h, w, ic, oc, k, p, s = case
    rng = np.random.default_rng(ic)
    # whole quarters: exact in both types, and so are the products and the sums of a few thousand of them in fp32
    x, wt, bias = (rng.integers(-8, 9, sh).astype(np.float32) / 4 for sh in ((n, h, w, ic), (oc, k, k, ic), (oc,)))
    pad = (p, p - (h + 2 * p - k) % s, p, p - (w + 2 * p - k) % s)
    want = oracle.conv2d("f64", *(v.astype(np.float64) for v in (x, wt, bias)), pad, (s, s), (1, 1))
    if dtype == capi.FP16:
        args = [v.astype(np.float16) for v in (x, wt, bias)]
    else:
        args = [(v.view(np.uint32) >> 16).astype(np.uint16) for v in (x, wt, bias)]
    got, st = gpu_ops.conv2d(ctx, *args, pad, (s, s), dtype=dtype)
    assert st == capi.VALID
    if dtype == capi.BF16:
        got = (got.astype(np.uint32) << 16).view(np.float32)
    # the sum is exact, so one rounding of the result is all there is: half a unit in the last place
    ulp = 2.0 ** -11 if dtype == capi.FP16 else 2.0 ** -8
    assert np.all(np.abs(got.astype(np.float64) - want) <= ulp * np.abs(want))
