"""MATMUL of any size and alignment: the kernel that splits K over waves at the edges of its tiles (32 x 64), blocks (64 bytes of K)
and shares, the last bytes of the operands, and the aligned copies behind large products."""
import numpy as np
import pytest

import cases
import dot_product_check as dp
import gpu_ops
import oracle
from reference_model_amd import Context, capi

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = Context(0)
    yield c
    c.close()


SHAPES = [  # n, h, c, w
    (1, 1, 1, 1), (1, 32, 64, 64), (2, 33, 65, 65), (3, 31, 63, 7), (1, 5, 130, 129), (2, 1, 1000, 70), (1, 64, 2049, 33),
    (9, 100, 200, 100), (40, 70, 31, 190), (1, 3, 5000, 8), (1, 40, 17, 1030), (4, 300, 66, 300),
]


@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("zps", [(0, 0), (-128, 127), (5, 0), (0, -3)])
def test_int8_of_any_size(ctx, shape, zps):
    n, h, c, w = shape
    rng = np.random.default_rng(h * c + w)
    a, b = rng.integers(-128, 128, (n, h, c)).astype(np.int8), rng.integers(-128, 128, (n, c, w)).astype(np.int8)
    got, st = gpu_ops.matmul(ctx, a, b, *zps)
    assert st == capi.VALID and ctx.last_kernel == "matmul_ragged_i8"
    assert np.array_equal(got, oracle.matmul("i8", a, b, *zps))


@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("kind", ["fp16", "bf16"])
def test_floating_point_of_any_size(ctx, shape, kind):
    n, h, c, w = shape
    rng = np.random.default_rng(h * c + w)
    a, b = rng.normal(0, 1, (n, h, c)).astype(np.float32), rng.normal(0, 1, (n, c, w)).astype(np.float32)
    if kind == "fp16":
        a, b, dtype = a.astype(np.float16), b.astype(np.float16), capi.FP16
        af, bf = a.astype(np.float64), b.astype(np.float64)
    else:
        a, b, dtype = cases.float_to_bf16_bits(a), cases.float_to_bf16_bits(b), capi.BF16
        af, bf = cases.bf16_bits_to_float(a).astype(np.float64), cases.bf16_bits_to_float(b).astype(np.float64)
    got, st = gpu_ops.matmul(ctx, a, b, dtype=dtype)
    assert st == capi.VALID and ctx.last_kernel == "matmul_ragged_" + {"fp16": "f16", "bf16": "bf16"}[kind]
    assert dp.check(got, np.matmul(af, bf), np.matmul(np.abs(af), np.abs(bf)), "fp32", dp.kernel_size_bound(c, "fp32", has_bias=False))["ok"]


def test_nothing_beyond_an_operand_enters_the_sums(ctx):
    """infinities and NaN right behind the rows and the end of both operands leave the results alone"""
    h, c, w = 33, 37, 67
    rng = np.random.default_rng(2)
    a, b = rng.normal(0, 1, (2, h, c)).astype(np.float16), rng.normal(0, 1, (2, c, w)).astype(np.float16)
    pad = np.array([np.inf, np.nan] * 64, np.float16)
    da, db = ctx.upload(np.concatenate([a.ravel(), pad])), ctx.upload(np.concatenate([b.ravel(), pad]))
    a[1, 0, 0], b[1, 0, 0] = np.inf, np.nan      # behind the first batch's operands
    da = ctx.upload(np.concatenate([a.ravel(), pad]))
    db = ctx.upload(np.concatenate([b.ravel(), pad]))
    out = ctx.empty((2, h, w), capi.FP32)
    ctx.matmul(capi.FP16, 2, h, c, w, da, db, 0, 0, out)
    assert ctx.sync() == capi.VALID
    want = np.matmul(a[0].astype(np.float64), b[0].astype(np.float64))
    assert np.allclose(out.numpy()[0], want, rtol=1e-4, atol=1e-4)


@pytest.mark.parametrize("shape", [(1, 1300, 1301, 1303), (2, 1100, 960, 1003), (1, 1400, 1217, 1344)])
def test_large_products_on_aligned_copies(ctx, shape):
    n, h, c, w = shape
    rng = np.random.default_rng(h)
    a, b = rng.integers(-128, 128, (n, h, c)).astype(np.int8), rng.integers(-128, 128, (n, c, w)).astype(np.int8)
    got, st = gpu_ops.matmul(ctx, a, b, 7, -9)
    assert st == capi.VALID and ctx.last_kernel == "matmul_pad_gemm_i8"
    assert np.array_equal(got, np.matmul(a.astype(np.float64) - 7, b.astype(np.float64) + 9).astype(np.int64).astype(np.int32))
    x, y = (a / 64).astype(np.float16), (b / 64).astype(np.float16)
    got, st = gpu_ops.matmul(ctx, x, y, dtype=capi.FP16)
    assert st == capi.VALID and ctx.last_kernel == "matmul_pad_gemm_f16"
    x, y = x.astype(np.float64), y.astype(np.float64)
    assert dp.check(got, np.matmul(x, y), np.matmul(np.abs(x), np.abs(y)), "fp32", dp.kernel_size_bound(c, "fp32", has_bias=False))["ok"]
