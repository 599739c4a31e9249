"""GPU parity of the streaming-patch CONV2D kernel (16-bit floats with taps, int8 with the fused RESCALE): slices of channels whole and cut, windows of two taps and
more, ragged rows, images and output channels.  Operands are small whole numbers, so that every sum is exact in fp32 and a
result has one right value in every type."""
import numpy as np
import pytest

import cases
import gpu_ops
import oracle
from reference_model_amd import Context, capi

pytestmark = pytest.mark.gpu

SHAPES = [  # n, ih, iw, ic, oc, kh, kw, pad, stride, dilation
    (16, 28, 28, 256, 64, 3, 3, (1, 1, 1, 1), (1, 1), (1, 1)),
    (10, 28, 30, 200, 56, 3, 3, (1, 1, 1, 1), (1, 1), (1, 1)),     # channels of no whole slices, output channels cut
    (12, 30, 28, 520, 128, 1, 3, (0, 0, 1, 1), (1, 1), (1, 1)),    # three taps: the next patch stored in a slice's second stage
    (24, 21, 23, 448, 136, 3, 1, (1, 1, 0, 0), (1, 1), (1, 1)),
    (9, 33, 41, 128, 64, 5, 5, (2, 2, 2, 2), (1, 1), (1, 1)),
    (12, 14, 14, 384, 264, 3, 3, (1, 1, 1, 1), (1, 1), (1, 1)),
    (14, 24, 28, 176, 56, 3, 3, (2, 2, 2, 2), (1, 1), (2, 2)),     # dilation
    (16, 29, 29, 328, 240, 3, 3, (1, 1, 1, 1), (2, 2), (1, 1)),    # stride
    (27, 40, 40, 264, 40, 3, 3, (1, 1, 1, 1), (1, 1), (1, 1)),     # more than 128 pixels a tile, the last rows of an image fewer
    (2, 60, 111, 256, 48, 3, 3, (1, 1, 1, 1), (1, 1), (1, 1)),     # a row a tile
    (16, 14, 14, 512, 512, 3, 3, (1, 1, 1, 1), (1, 1), (1, 1)),
]


@pytest.fixture(scope="module")
def ctx():
    c = Context(0)
    yield c
    c.close()


@pytest.mark.parametrize("kind", ["fp16", "bf16"])
@pytest.mark.parametrize("shape", SHAPES)
def test_small_whole_numbers(ctx, kind, shape):
    n, ih, iw, ic, oc, kh, kw, pad, stride, dil = shape
    rng = np.random.default_rng(ic + oc)
    x = rng.integers(-2, 3, (n, ih, iw, ic)).astype(np.int8)
    w = rng.integers(-2, 3, (oc, kh, kw, ic)).astype(np.int8)
    bias = rng.integers(-9, 10, oc).astype(np.int32)
    want = cases.conv2d_exact_blas(x, w, bias, pad, stride, dil)
    if kind == "fp16":
        got, st = gpu_ops.conv2d(ctx, *(v.astype(np.float16) for v in (x, w, bias)), pad, stride, dil, dtype=capi.FP16)
        want = want.astype(np.float16)
    else:
        got, st = gpu_ops.conv2d(ctx, *(cases.float_to_bf16_bits(v.astype(np.float32)) for v in (x, w, bias)), pad, stride, dil, dtype=capi.BF16)
        want = cases.float_to_bf16_bits(want.astype(np.float32))
    assert st == capi.VALID
    print(shape, ctx.last_kernel)
    assert np.array_equal(got, want)


@pytest.mark.parametrize("shape", [(7, 14, 21, 200, 288), (16, 28, 28, 256, 64)])
def test_infinite_weights_outside_the_image(ctx, shape):
    """a tap outside the image adds nothing, also where its weight is infinite or NaN"""
    n, ih, iw, ic, oc = shape
    rng = np.random.default_rng(3)
    x = rng.integers(1, 4, (n, ih, iw, ic)).astype(np.float16)
    w = rng.integers(-2, 3, (oc, 3, 3, ic)).astype(np.float16)
    w[:, :, :, 0] = 1
    plain = w.copy()
    w[3, 0, 0, 5], w[oc - 1, 1, 2, ic - 1], w[8, 2, 2, 1] = np.inf, np.nan, -np.inf    # the top left tap, right, bottom right
    b = np.zeros(oc, np.float16)
    want, _ = gpu_ops.conv2d(ctx, x, plain, b, (1, 1, 1, 1), dtype=capi.FP16)
    got, st = gpu_ops.conv2d(ctx, x, w, b, (1, 1, 1, 1), dtype=capi.FP16)
    assert st == capi.VALID
    # without a channel of the tap that lies outside: the results of finite weights there
    one = [c for c in range(oc) if c not in (3, 8, oc - 1)]
    assert np.array_equal(got[..., one], want[..., one])
    assert np.array_equal(got[:, 0, :, 3], want[:, 0, :, 3]) and np.array_equal(got[:, :, 0, 3], want[:, :, 0, 3])
    assert np.isposinf(got[:, 1:, 1:, 3]).all()
    assert np.array_equal(got[:, -1, :, 8], want[:, -1, :, 8]) and np.isneginf(got[:, :-1, :-1, 8]).all()
    assert np.array_equal(got[:, :, -1, oc - 1], want[:, :, -1, oc - 1]) and np.isnan(got[:, :, :-1, oc - 1]).all()


I8_SHAPES = [  # the same for int8 with the fused RESCALE
    (14, 30, 30, 592, 96, 3, 3, (1, 1, 1, 1), (1, 1), (1, 1)),
    (32, 13, 10, 480, 136, 3, 3, (1, 1, 1, 1), (1, 1), (1, 1)),
    (9, 33, 41, 256, 72, 5, 5, (2, 2, 2, 2), (1, 1), (1, 1)),
    (12, 30, 28, 768, 128, 1, 3, (0, 0, 1, 1), (1, 1), (1, 1)),
    (27, 40, 40, 400, 40, 3, 3, (1, 1, 1, 1), (1, 1), (1, 1)),
    (16, 29, 29, 512, 264, 3, 3, (1, 1, 1, 1), (2, 2), (1, 1)),
]


@pytest.mark.parametrize("in_zp, double_round, clamp", [(0, True, None), (-128, False, (-100, 90)), (17, True, (5, 127))])
@pytest.mark.parametrize("shape", I8_SHAPES)
def test_int8_rescale(ctx, shape, in_zp, double_round, clamp):
    n, ih, iw, ic, oc, kh, kw, pad, stride, dil = shape
    rng = np.random.default_rng(ic + oc + in_zp)
    x = rng.integers(-128, 128, (n, ih, iw, ic)).astype(np.int8)
    w = rng.integers(-128, 128, (oc, kh, kw, ic)).astype(np.int8)
    bias = rng.integers(-(1 << 18), 1 << 18, oc).astype(np.int32)
    mult = rng.integers(1 << 30, (1 << 31) - 1, oc).astype(np.int32)
    shift = rng.integers(41, 45, oc).astype(np.int8)
    mode = capi.ROUND_DOUBLE if double_round else capi.ROUND_SINGLE
    want, wst = oracle.rescale(cases.conv2d_exact_blas(x, w, bias, pad, stride, dil, in_zp), mult, shift, out_zp=5, rounding_mode=mode)
    if clamp:
        want = oracle.clamp(want, *clamp)
    got, st = gpu_ops.conv2d(ctx, x, w, bias, pad, stride, dil, in_zp=in_zp, rescale=dict(mult=mult, shift=shift, out_zp=5, rounding_mode=mode), clamp=clamp)
    assert st == wst == capi.VALID
    assert np.array_equal(got, want)


# Which of them the kernel has, so that a change of its rule does not leave the tests above to others.  The window of one column on 448 channels
# (161 pixels a tile) is the GEMM kernel's and the strided int8 layer on 512 channels a split reduction's; shapes that stay stand in for them.
ELSEWHERE = [(24, 21, 23, 448, 136, 3, 1, (1, 1, 0, 0), (1, 1), (1, 1)), (16, 29, 29, 512, 264, 3, 3, (1, 1, 1, 1), (2, 2), (1, 1))]


@pytest.mark.parametrize("kind", ["fp16", "bf16"])
@pytest.mark.parametrize("shape", [s for s in SHAPES if s not in ELSEWHERE] + [(24, 42, 23, 448, 56, 3, 1, (1, 1, 0, 0), (1, 1), (1, 1))])
def test_which_kernel(ctx, kind, shape):
    test_small_whole_numbers(ctx, kind, shape)
    assert ctx.last_kernel == ("conv2d_planes_f16" if kind == "fp16" else "conv2d_planes_bf16")


@pytest.mark.parametrize("in_zp", [0, 17])
@pytest.mark.parametrize("shape", [s for s in I8_SHAPES if s not in ELSEWHERE] + [(16, 29, 29, 640, 264, 3, 3, (1, 1, 1, 1), (2, 2), (1, 1))])
def test_which_kernel_int8(ctx, shape, in_zp):
    test_int8_rescale(ctx, shape, in_zp, True, None)
    assert ctx.last_kernel == "conv2d_planes_i8_rescale"


@pytest.mark.parametrize("kind, shape, kernel", [  # n, h, w, ic, oc, k, stride
    # up to 32 output channels on tiles of more than 128 pixels: the patch kernel's, but for long rows of 16-bit floats
    ("int8", (21, 48, 48, 192, 32, 3, 1), "conv2d_mfma_i8_rescale"),
    ("int8", (13, 34, 89, 192, 8, 3, 1), "conv2d_mfma_i8_rescale"),
    ("bf16", (16, 55, 55, 96, 32, 3, 1), "conv2d_mfma_bf16"),
    ("fp16", (9, 71, 71, 80, 32, 3, 1), "conv2d_mfma_f16"),
    ("fp16", (5, 52, 22, 512, 16, 3, 1), "conv2d_taps_f16"),
    ("fp16", (31, 52, 22, 512, 16, 3, 1), "conv2d_planes_f16"),
    ("bf16", (16, 55, 55, 96, 40, 3, 1), "conv2d_planes_bf16"),
    # a slice cut off, and the split reductions' last round of tiles four fifths full; less full, or whole slices
    ("bf16", (9, 14, 61, 136, 328, 3, 2), "conv2d_taps_bf16"),
    ("fp16", (11, 23, 8, 88, 216, 5, 1), "conv2d_taps_f16"),
    ("fp16", (4, 47, 8, 144, 320, 3, 1), "conv2d_taps_f16"),
    ("fp16", (12, 96, 21, 176, 96, 3, 2), "conv2d_planes_f16"),
    ("fp16", (3, 76, 20, 128, 104, 3, 1), "conv2d_planes_f16"),
])
def test_layers_it_leaves(ctx, kind, shape, kernel):
    n, h, w, ic, oc, k, s = shape
    p = k // 2
    pad = (p, p - (h + 2 * p - k) % s, p, p - (w + 2 * p - k) % s)
    case = (n, h, w, ic, oc, k, k, pad, (s, s), (1, 1))
    if kind == "int8":
        test_int8_rescale(ctx, case, 17, True, None)
    else:
        test_small_whole_numbers(ctx, kind, case)
    assert ctx.last_kernel == kernel
