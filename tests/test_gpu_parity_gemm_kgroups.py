"""GPU parity of the GEMM kernel where two groups of waves share the K-steps of a block (128 x 128 tiles, blocks requested in
pairs, taps or zero points): block counts round the ring's length, odd and even, ragged tiles.  Operands are small whole
numbers, so that every sum is exact in fp32 and a result has one right value in every type."""
import numpy as np
import pytest

import cases
import gpu_ops
from reference_model_amd import Context, capi

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = Context(0)
    c.set_kernel_choice(capi.KERNEL_GEMM)
    yield c
    c.close()


@pytest.mark.parametrize("kind", ["int8", "fp16", "bf16"])
@pytest.mark.parametrize("blocks, kh, kw", [(33, 1, 3), (34, 2, 1), (39, 1, 3), (40, 2, 2), (45, 3, 3), (56, 2, 4)])
def test_taps(ctx, kind, blocks, kh, kw):
    channels = blocks // (kh * kw) * (64 if kind == "int8" else 32)
    rng = np.random.default_rng(blocks)
    x = rng.integers(-2, 3, (6, 63, 65, channels)).astype(np.int8)
    w = rng.integers(-2, 3, (130, kh, kw, channels)).astype(np.int8)
    bias = rng.integers(-9, 10, 130).astype(np.int32)
    pad, stride, dil = (kh // 2, kh - 1 - kh // 2, kw // 2, kw - 1 - kw // 2), (2, 2), (1, 1)
    zps = (3, -2) if kind == "int8" else (0, 0)
    want = cases.conv2d_exact_blas(x, w, bias, pad, stride, dil, *zps)
    if kind == "int8":
        got, st = gpu_ops.conv2d(ctx, x, w, bias, pad, stride, dil, *zps)
    elif kind == "fp16":
        got, st = gpu_ops.conv2d(ctx, *(v.astype(np.float16) for v in (x, w, bias)), pad, stride, dil, dtype=capi.FP16)
        want = want.astype(np.float16)
    else:
        got, st = gpu_ops.conv2d(ctx, *(cases.float_to_bf16_bits(v.astype(np.float32)) for v in (x, w, bias)), pad, stride, dil, dtype=capi.BF16)
        want = cases.float_to_bf16_bits(want.astype(np.float32))
    assert st == capi.VALID and ctx.last_kernel == {"int8": "gemm_mfma_i8", "fp16": "gemm_mfma_f16", "bf16": "gemm_mfma_bf16"}[kind]
    assert np.array_equal(got, want)


@pytest.mark.parametrize("blocks", [33, 34, 39, 40, 41])
@pytest.mark.parametrize("w", [336, 340])    # the second operand read as it lies; from a transposed copy
def test_matmul_zero_points(ctx, blocks, w):
    rng = np.random.default_rng(blocks + w)
    a = rng.integers(-128, 128, (3, 333, 64 * blocks)).astype(np.int8)
    b = rng.integers(-128, 128, (3, 64 * blocks, w)).astype(np.int8)
    got, st = gpu_ops.matmul(ctx, a, b, -7, 100)
    assert st == capi.VALID and ctx.last_kernel == ("matmul_gemm_i8" if w % 16 == 0 else "matmul_tgemm_i8")
    assert np.array_equal(got, np.matmul(a.astype(np.float64) + 7, b.astype(np.float64) - 100).astype(np.int64))
