"""CONV2D on 16-bit floats with infinite and NaN weights under taps that fall outside the image, which add nothing in the reference
(tensor_ops.cpp:845-852), and with NaN in the image: results of other channels keep their bits, and a NaN image costs no sums."""
import time

import numpy as np
import pytest

import cases
import gpu_ops
from reference_model_amd import Context, capi

pytestmark = pytest.mark.gpu

CASES = [  # kernel, kernel choice, n, ih, iw, ic, oc, k, stride, dilation
    ("conv2d_planes_f16", 0, 7, 14, 21, 200, 288, 3, 1, 1),
    ("conv2d_planes_bf16", 0, 16, 28, 28, 256, 64, 3, 1, 1),
    ("conv2d_planes_f16", 0, 16, 29, 29, 328, 240, 3, 2, 1),
    ("gemm_mfma_f16_patch", 0, 4, 28, 28, 224, 256, 3, 1, 1),
    ("gemm_mfma_bf16_patch", 0, 16, 26, 26, 256, 512, 1, 1, 1),    # one tap and a border: windows that lie outside altogether
    ("gemm_mfma_bf16", 0, 64, 7, 7, 512, 512, 3, 1, 1),
    ("gemm_mfma_f16", 0, 32, 56, 56, 64, 128, 3, 2, 1),
    ("gemm_mfma_f16", 0, 16, 56, 56, 128, 100, 3, 1, 1),           # rows of no whole 16 bytes
    ("conv2d_mfma_f16", 0, 2, 28, 28, 256, 250, 3, 1, 1),
    ("conv2d_mfma_bf16", 0, 4, 100, 130, 128, 64, 3, 1, 1),
    ("conv2d_mfma_f16", 2, 2, 15, 13, 36, 72, 5, 1, 2),
    ("conv2d_mfma_bf16", 2, 1, 9, 9, 17, 24, 3, 1, 1),
    ("conv2d_slab_f16", 0, 8, 56, 56, 64, 64, 3, 1, 1),
    ("conv2d_slab_bf16", 0, 4, 29, 29, 48, 96, 3, 2, 1),
    ("conv2d_slab_f16", 4, 1, 9, 9, 32, 48, 3, 1, 1),              # half a block of channels
    ("conv2d_slab_bf16", 0, 8, 28, 28, 256, 128, 1, 1, 1),
    ("conv2d_taps_f16", 0, 15, 54, 65, 68, 64, 3, 1, 1),           # weights resident, two tiles of channels
    ("conv2d_taps_bf16", 0, 2, 79, 7, 88, 23, 3, 1, 1),
    ("conv2d_taps_f16", 0, 9, 31, 41, 240, 32, 3, 2, 1),           # K split
    ("conv2d_taps_bf16", 0, 2, 14, 13, 200, 40, 5, 1, 1),
    ("conv2d_taps_f16", 0, 2, 12, 11, 45, 48, 3, 1, 2),            # rows between words
]


@pytest.fixture(scope="module", params=CASES, ids=lambda c: "-".join(str(v) for v in c))
def layer(request):
    kernel, choice, n, ih, iw, ic, oc, k, s, d = request.param
    rng = np.random.default_rng(ic + oc)
    half = np.float16 if "_f16" in kernel else None
    x, w, b = rng.normal(0, 1, (n, ih, iw, ic)), rng.normal(0, 0.05, (oc, k, k, ic)), rng.normal(0, 1, oc)
    x, w, b = (v.astype(np.float16) if half else cases.float_to_bf16_bits(v.astype(np.float32)) for v in (x, w, b))
    p = max(d * (k // 2), 1)
    ends = [p - (size + 2 * p - d * (k - 1) - 1) % s for size in (ih, iw)]
    ctx = Context(0)
    ctx.set_kernel_choice(choice)

    def run(x, w):
        got, st = gpu_ops.conv2d(ctx, x, w, b, (p, ends[0], p, ends[1]), (s, s), (d, d), dtype=capi.FP16 if half else capi.BF16)
        assert st == capi.VALID and ctx.last_kernel == kernel
        return got

    def device(x):
        code, shape = capi.FP16 if half else capi.BF16, layer["plain"].shape
        desc = ctx.conv_desc(code, code, x.shape, oc, k, k, shape[1:3], (p, ends[0], p, ends[1]), (s, s), (d, d), oc)
        tensors = [ctx.upload(v, code) for v in (x, w, b)] + [ctx.empty(shape, code, x.dtype)]
        return tensors, lambda: ctx.conv2d(desc, *tensors[:3], 0, 0, tensors[3])
    wide = (lambda v: v.astype(np.float64)) if half else (lambda v: (v.astype(np.uint32) << 16).view(np.float32).astype(np.float64))
    # which results have tap (ky, kx) inside the image: [ky][oh], [kx][ow]
    rows, cols = ([[0 <= o * s - p + t * d < size for o in range(length)] for t in range(k)] for size, length in zip((ih, iw), run(x, w).shape[1:3]))
    bits = {"inf": np.float16(np.inf), "-inf": np.float16(-np.inf), "nan": np.float16(np.nan)} if half else {"inf": 0x7f80, "-inf": 0xff80, "nan": 0x7fc0}
    layer = dict(ctx=ctx, device=device, run=run, x=x, w=w, plain=run(x, w), wide=wide, rows=np.array(rows), cols=np.array(cols), bits=bits, s=s, d=d, p=p, ulp=2.0 ** -10 if half else 2.0 ** -7)
    yield layer
    ctx.close()


def test_weights_that_are_no_numbers(layer):
    w, (oc, k, _, ic) = layer["w"].copy(), layer["w"].shape
    odd = {3: (0, 0, 5, "inf"), 8: (k - 1, k - 1, 1, "-inf"), 20: (0, k - 1, ic - 1, "nan"), oc - 1: (k // 2, 0, 9, "inf")}    # channel: the tap, its input channel
    for c, (ky, kx, i, what) in odd.items():
        w[c, ky, kx, i] = layer["bits"][what]
    got, plain = layer["run"](layer["x"], w), layer["plain"]
    same = [c for c in range(oc) if c not in odd]
    assert np.array_equal(got[..., same].view(np.uint16), plain[..., same].view(np.uint16))
    met_outside = False
    reach = np.abs(layer["wide"](layer["x"])).max()
    for c, (ky, kx, i, what) in odd.items():
        inside = layer["rows"][ky][:, None] & layer["cols"][kx][None, :]
        assert inside.any()
        met_outside |= not inside.all()
        g, p = layer["wide"](got[..., c]), layer["wide"](plain[..., c])
        assert not np.isfinite(g[:, inside]).any()
        # the sums without the tap, in another order: K roundings of 2^-24 of the absolute products on either side, and two of the result
        terms = layer["w"][c].size
        slack = 2 * terms * 2.0 ** -24 * reach * np.abs(layer["wide"](layer["w"][c])).sum()
        assert np.all(np.abs(g - p)[:, ~inside] <= layer["ulp"] * np.abs(p)[:, ~inside] + slack)
    assert met_outside


def test_a_nan_pixel(layer):
    x = layer["x"].copy()
    x[0, 0, 0, 7] = layer["bits"]["nan"]
    got, plain = layer["run"](x, layer["w"]), layer["plain"]
    met = np.isnan(layer["wide"](got))
    reached = [np.any([layer[axis][t] & (np.arange(len(layer[axis][t])) * layer["s"] + t * layer["d"] == layer["p"]) for t in range(len(layer[axis]))], axis=0) for axis in ("rows", "cols")]
    assert np.array_equal(met[0], np.broadcast_to((reached[0][:, None] & reached[1][None, :])[..., None], met[0].shape)) and met.any() and not met[1:].any()
    assert np.array_equal(got[~met].view(np.uint16), plain[~met].view(np.uint16))


def test_a_nan_image_costs_no_sums(layer):
    """A result that is NaN through its window costs a look at the weights; summed again one product after the other it took 150 to 230 times as long."""
    def seconds(x):
        tensors, call = layer["device"](x)
        call(), layer["ctx"].sync()
        start = time.perf_counter()
        for _ in range(20):
            call()
        assert layer["ctx"].sync() == capi.VALID
        taken, got = time.perf_counter() - start, tensors[-1].numpy()
        for t in tensors:
            t.free()
        return taken, got
    finite, _ = seconds(layer["x"])
    nan, got = seconds(np.full_like(layer["x"], layer["bits"]["nan"]))
    print("us a call, finite / NaN:", finite / 20e-6, nan / 20e-6)
    reached = layer["rows"].any(axis=0)[:, None] & layer["cols"].any(axis=0)[None, :]    # (a window that lies outside altogether: the bias)
    assert np.array_equal(np.isnan(layer["wide"](got)), np.broadcast_to(reached[None, :, :, None], got.shape)) and nan < 4 * finite
