"""MATMUL by the kernel that splits K over waves: tiles of 32 columns, the last bytes of the operands wherever a load begins, operands of
less than one load, and the eighths of the grid that share an L2."""
import time

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
    (1, 33, 1025, 31), (2, 32, 1056, 65), (3, 7, 2047, 97),    # sixteen waves a tile: 32 columns, ragged every way
    (7, 40, 1100, 500),                                         # 112 tiles of 64: the last of them; one more below
    (1, 3600, 1030, 3),
    (5, 1, 3, 5), (1, 2, 4, 1), (1, 1, 7, 2),                   # an operand of less than 16 bytes
    (2, 5, 9, 3), (1, 4, 40, 1), (3, 33, 8, 9),                 # rows shorter than a load
    (9, 100, 33, 70), (13, 65, 70, 129),                        # a grid that is no multiple of eight
]


@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("kind", ["int8", "fp16", "bf16"])
def test_edges_of_the_split_kernel(ctx, shape, kind):
    n, h, c, w = shape
    rng = np.random.default_rng(h * c + w)
    if kind == "int8":
        a, b = rng.integers(-128, 128, (n, h, c)).astype(np.int8), rng.integers(-128, 128, (n, c, w)).astype(np.int8)
        got, st = gpu_ops.matmul(ctx, a, b, -7, 100)
        assert st == capi.VALID and ctx.last_kernel == "matmul_ragged_i8" and np.array_equal(got, oracle.matmul("i8", a, b, -7, 100))
        return
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


@pytest.mark.parametrize("shape", [(2, 33, 1037, 67), (1, 1, 1, 1), (2, 3, 5, 2), (1, 40, 2000, 30)])
def test_nothing_around_the_operands_is_used(ctx, shape):
    """infinities and NaN before and behind both operands, on addresses of no alignment"""
    n, h, c, w = shape
    rng = np.random.default_rng(3)
    a, b = rng.normal(0, 1, (n, h, c)).astype(np.float16), rng.normal(0, 1, (n, c, w)).astype(np.float16)
    pad = np.array([np.inf, np.nan] * 32, np.float16)
    da, db = (ctx.upload(np.concatenate([pad[:3], v.ravel(), pad])) for v in (a, b))
    out = ctx.empty((n, h, w), capi.FP32)
    ctx.matmul(capi.FP16, n, h, c, w, da.ptr + 6, db.ptr + 6, 0, 0, out)
    assert ctx.sync() == capi.VALID
    af, bf = a.astype(np.float64), b.astype(np.float64)
    assert dp.check(out.numpy(), np.matmul(af, bf), np.matmul(np.abs(af), np.abs(bf)), "fp32", dp.kernel_size_bound(c, "fp32", has_bias=False))["ok"]


def test_rows_beyond_32_bit_offsets(ctx):
    """rows just below and just above what 32 rows' offsets reach in 32 bits: the same results, at the same rate (element by element the second
    took five times as long)"""
    rng = np.random.default_rng(1)
    border = (2 ** 31 - 1) // 33
    a, b = (rng.integers(-1, 2, border + 64).astype(np.int8) for _ in range(2))
    da, db, out = ctx.upload(a), ctx.upload(b), ctx.empty((1,), capi.INT32)
    took = []
    for c in (border - 5, border + 5):
        best = 1e9
        for _ in range(3):
            t0 = time.perf_counter()
            ctx.matmul(capi.INT8, 1, 1, c, 1, da.ptr, db.ptr, 1, -1, out)
            assert ctx.sync() == capi.VALID and ctx.last_kernel == "matmul_ragged_i8"
            best = min(best, time.perf_counter() - t0)
        took.append(best)
        assert out.numpy()[0] == int(np.dot(a[:c].astype(np.int64) - 1, b[:c].astype(np.int64) + 1))
    assert took[1] < 2 * took[0]
