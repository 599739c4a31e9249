"""The GEMM kernel's results of every row length: rows of whole 128-byte lines, of whole 16-byte pieces, of words and of single elements, at
the edges of its tiles, for the products of MATMUL and the layers of CONV2D."""
import numpy as np
import pytest

import cases
import dot_product_check as dp
import gpu_ops
from reference_model_amd import Context, capi

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = Context(0)
    c.set_kernel_choice(capi.KERNEL_GEMM)
    yield c
    c.close()


def narrow(v, kind):
    """(device operand, its value in float64, the data type)"""
    if kind == "fp16":
        v = v.astype(np.float16)
        return v, v.astype(np.float64), capi.FP16
    v = cases.float_to_bf16_bits(v.astype(np.float32))
    return v, cases.bf16_bits_to_float(v).astype(np.float64), capi.BF16


@pytest.mark.parametrize("shape", [(3, 300, 64, 136), (3, 257, 160, 168), (2, 130, 96, 104),    # whole pieces; tiles of 128 x 128
                                   (3, 1100, 320, 1112), (6, 1030, 256, 1048),                    # larger tiles
                                   (3, 300, 64, 301), (3, 257, 96, 130), (4, 1000, 128, 1003)])   # words, on a transposed copy
@pytest.mark.parametrize("kind", ["int8", "fp16", "bf16"])
def test_matmul_rows(ctx, shape, kind):
    n, h, c, w = shape
    rng = np.random.default_rng(w)
    if kind == "int8":
        c = -(-c // 64) * 64
        for za, zb in ((0, 0), (-9, 4)):
            for cols in (w, -(-w // 16) * 16):
                a, b = rng.integers(-128, 128, (n, h, c)).astype(np.int8), rng.integers(-128, 128, (n, c, cols)).astype(np.int8)
                got, st = gpu_ops.matmul(ctx, a, b, za, zb)
                assert st == capi.VALID and "gemm" in ctx.last_kernel
                assert np.array_equal(got, np.matmul(a.astype(np.float64) - za, b.astype(np.float64) - zb).astype(np.int64))
        return
    (a, af, dtype), (b, bf, _) = (narrow(rng.normal(0, 1, s), kind) for s in ((n, h, c), (n, c, w)))
    got, st = gpu_ops.matmul(ctx, a, b, dtype=dtype)
    assert st == capi.VALID and "gemm" in ctx.last_kernel
    assert dp.check(got, np.matmul(af, bf), np.matmul(np.abs(af), np.abs(bf)), "fp32", dp.kernel_size_bound(c, "fp32", has_bias=False))["ok"]


@pytest.mark.parametrize("case", [(9, 30, 64, 1, (64, 72, 136, 132, 134, 131)),       # pointwise: tiles of 128 channels
                                  (24, 40, 64, 1, (512, 520, 518, 517)),              # of 256
                                  (12, 28, 128, 3, (192, 200, 196, 195, 129))])       # taps, and the patch form
@pytest.mark.parametrize("kind", ["fp16", "bf16"])
def test_conv2d_rows(ctx, case, kind):
    n, hw, ic, k, channels = case
    rng = np.random.default_rng(ic)
    x, xf, dtype = narrow(rng.normal(0, 1, (n, hw, hw, ic)), kind)
    for oc in channels:
        (w, wf, _), (b, bf, _) = narrow(rng.normal(0, 1 / np.sqrt(k * k * ic), (oc, k, k, ic)), kind), narrow(rng.normal(0, 1, oc), kind)
        pad = (k // 2,) * 4
        got, st = gpu_ops.conv2d(ctx, x, w, b, pad, dtype=dtype)
        assert st == capi.VALID and "gemm" in ctx.last_kernel
        got = got.astype(np.float64) if kind == "fp16" else cases.bf16_bits_to_float(got).astype(np.float64)
        pick = [0, n // 2, n - 1]    # (images)
        p = np.pad(xf[pick], ((0, 0), (k // 2, k // 2), (k // 2, k // 2), (0, 0)))
        want = mag = 0.0
        for ky in range(k):
            for kx in range(k):
                v = p[:, ky:ky + hw, kx:kx + hw].reshape(-1, ic)
                want, mag = want + v @ wf[:, ky, kx].T, mag + np.abs(v) @ np.abs(wf[:, ky, kx]).T
        assert dp.check(got[pick].reshape(want.shape), want + bf, mag + np.abs(bf), kind, dp.kernel_size_bound(k * k * ic, kind))["ok"]
