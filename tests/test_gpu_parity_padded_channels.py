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


CASES = {  # n, h, w, ic, oc, k, pad, stride: the kernel of the int8 layer
    # copies padded first
    (6, 45, 45, 65, 24, 3, 1, 1): "conv2d_taps_i8",      # one byte past a piece
    (10, 47, 49, 31, 8, 5, 2, 1): "conv2d_mfma_i8",      # one short of a step
    (40, 57, 57, 33, 131, 1, 0, 1): "gemm_mfma_i8",
    (3, 11, 5, 131, 40, 3, 1, 2): "conv2d_ksplit_i8",
    (6, 40, 41, 207, 64, 2, 0, 1): "conv2d_ksplit_i8",
    (16, 16, 16, 72, 72, 3, 1, 1): "conv2d_ksplit_i8",    # whole words
    (4, 53, 53, 80, 80, 3, 1, 1): "conv2d_slab_i8",
    (1, 10, 10, 245, 16, 3, 1, 1): "conv2d_ksplit_patch_i8",    # padded to 256: both operands in LDS
    # smaller ones, and few channels in short reductions: one launch, as they lie
    (11, 45, 45, 17, 24, 3, 1, 1): "conv2d_taps_i8",
    (10, 47, 49, 31, 8, 3, 1, 1): "conv2d_taps_i8",
    (20, 57, 57, 65, 24, 1, 0, 1): "conv2d_taps_i8",
    (1, 7, 9, 17, 24, 3, 1, 1): "conv2d_taps_i8",
    (2, 9, 7, 31, 8, 3, 1, 1): "conv2d_taps_i8",
    (1, 8, 8, 33, 13, 1, 0, 1): "conv2d_taps_i8",
    (1, 8, 8, 65, 24, 1, 0, 1): "conv2d_taps_i8",
    (1, 6, 6, 207, 64, 2, 0, 1): "conv2d_taps_i8",
    (2, 13, 13, 72, 72, 3, 1, 1): "conv2d_taps_i8",
    (2, 12, 12, 80, 80, 3, 1, 1): "conv2d_taps_i8",
}


@pytest.mark.parametrize("ic, oc, fused, kernel", [
    (17, 16, True, "conv2d_taps_i8_rescale"), (27, 32, True, "conv2d_taps_i8_rescale"), (45, 64, True, "conv2d_taps_i8_rescale"),
    (21, 20, True, "conv2d_taps_i8_rescale"), (17, 16, False, "conv2d_taps_i8"), (37, 8, False, "conv2d_taps_i8"),
    (7, 9, True, "conv2d_direct_i8_rescale"), (7, 9, False, "conv2d_direct_i8")])
def test_tiny_layers_stay_one_launch(ic, oc, fused, kernel):
    """the one-result-per-lane kernel or the one with split reductions reads the operands as they lie, without a copy in scratch memory"""
    rng = np.random.default_rng(ic)
    x, wt = rng.integers(-128, 128, (1, 9, 8, ic)).astype(np.int8), rng.integers(-128, 128, (oc, 1, 1, ic)).astype(np.int8)
    bias = rng.integers(-999, 999, oc).astype(np.int32)
    mult, shift = rng.integers(1 << 30, 1 << 31, oc).astype(np.int32), rng.integers(38, 43, oc).astype(np.int8)
    want = oracle.conv2d("i8", x, wt, bias, (0, 0, 0, 0), (1, 1), (1, 1), in_zp=5, w_zp=0)
    if fused:
        want, _ = oracle.rescale(want, mult, shift, out_zp=3)
    c = Context(0)
    try:
        got, st = gpu_ops.conv2d(c, x, wt, bias, in_zp=5, w_zp=0, rescale=dict(mult=mult, shift=shift, out_zp=3) if fused else None)
        assert st == capi.VALID and np.array_equal(got, want)
        assert c.last_kernel == kernel and c.workspace_bytes() == (0, 0)
    finally:
        c.close()


@pytest.mark.parametrize("case", CASES)
def test_only_large_or_odd_layers_are_copied(case):
    n, h, w, ic, oc, k, p, s = case
    pad = (p, p - (h + 2 * p - k) % s, p, p - (w + 2 * p - k) % s)
    c = Context(0)
    try:
        _, st = gpu_ops.conv2d(c, np.ones((n, h, w, ic), np.int8), np.ones((oc, k, k, ic), np.int8), np.zeros(oc, np.int32), pad, (s, s))
        copied = list(CASES).index(case) < 8
        assert st == capi.VALID and (c.workspace_bytes() != (0, 0)) == copied
    finally:
        c.close()


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
        assert st == capi.VALID and np.array_equal(got, want) and ctx.last_kernel == CASES[case]
        return
    mult, shift = rng.integers(1 << 30, 1 << 31, oc).astype(np.int32), rng.integers(38, 43, oc).astype(np.int8)
    want, wst = oracle.rescale(want, mult, shift, out_zp=3)
    got, st = gpu_ops.conv2d(ctx, x, wt, bias, pad, (s, s), in_zp=-11, w_zp=0, rescale=dict(mult=mult, shift=shift, out_zp=3))
    assert st == wst and np.array_equal(got, want) and len(np.unique(got)) > 20 and ctx.last_kernel == CASES[case] + "_rescale"


def test_pointwise_layer_on_copies():
    """many channels on more tiles than the kernel that reads as they lie has workgroups: copies, and the kernel that keeps its weights in registers"""
    n, h, w, ic, oc = 40, 20, 20, 65, 136
    rng = np.random.default_rng(3)
    x, wt = rng.integers(-128, 128, (n, h, w, ic)).astype(np.int8), rng.integers(-128, 128, (oc, 1, 1, ic)).astype(np.int8)
    bias = rng.integers(-9999, 9999, oc).astype(np.int32)
    mult, shift = rng.integers(1 << 30, 1 << 31, oc).astype(np.int32), rng.integers(38, 43, oc).astype(np.int8)
    want, wst = oracle.rescale(oracle.conv2d("i8", x, wt, bias, in_zp=-11, w_zp=0), mult, shift, out_zp=3)
    c = Context(0)
    try:
        got, st = gpu_ops.conv2d(c, x, wt, bias, in_zp=-11, w_zp=0, rescale=dict(mult=mult, shift=shift, out_zp=3))
        assert st == wst and np.array_equal(got, want) and len(np.unique(got)) > 20
        assert c.last_kernel == "conv2d_pointwise_i8_rescale" and c.workspace_bytes() != (0, 0)
    finally:
        c.close()


def test_padded_layer_with_its_sums_in_the_scratch_buffer():
    """a fused layer under precise-mode INEXACT_ROUND keeps its INT32 sums in the context's scratch buffer; the padded operands of
    the same call lie elsewhere"""
    n, h, w, ic, oc = 2, 12, 12, 131, 48
    rng = np.random.default_rng(8)
    x, wt = rng.integers(-128, 128, (n, h, w, ic)).astype(np.int8), rng.integers(-128, 128, (oc, 3, 3, ic)).astype(np.int8)
    bias, pad = rng.integers(-9999, 9999, oc).astype(np.int32), (1, 1, 1, 1)
    mult, shift = rng.integers(1 << 29, 1 << 30, oc).astype(np.int32), rng.integers(40, 44, oc).astype(np.int8)
    acc = oracle.conv2d("i8", x, wt, bias, pad, (1, 1), (1, 1), in_zp=-11, w_zp=0)
    want, wst = oracle.rescale(acc, mult, shift, out_zp=3, rounding_mode=capi.ROUND_INEXACT, inexact_mode=1)
    c = Context(0)
    try:
        c.set_precise_mode(True)
        for _ in range(2):
            got, st = gpu_ops.conv2d(c, x, wt, bias, pad, in_zp=-11, w_zp=0,
                                     rescale=dict(mult=mult, shift=shift, out_zp=3, rounding_mode=capi.ROUND_INEXACT))
            assert st == wst and np.array_equal(got, want) and len(np.unique(got)) > 20
        # the sums, and the padded operands of 160 channels
        assert c.workspace_bytes()[0] >= 4 * n * h * w * oc + 160 * (n * h * w + 9 * oc)
    finally:
        c.close()


@pytest.mark.parametrize("case", list(CASES) + [(1, 9, 9, 9, 16, 3, 1, 1), (1, 9, 9, 100, 40, 3, 1, 1), (2, 12, 12, 40, 64, 3, 1, 1)])
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
