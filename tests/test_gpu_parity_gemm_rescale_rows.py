"""The GEMM kernel's fused RESCALE results of every row length: whole 16-byte pieces, words and single elements, of both output types."""
import numpy as np
import pytest

import cases
import gpu_ops
import oracle
from reference_model_amd import Context, capi

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = Context(0)
    c.set_kernel_choice(capi.KERNEL_GEMM)
    yield c
    c.close()


@pytest.mark.parametrize("case", [(9, 30, 128, 1), (3, 70, 64, 1), (12, 28, 128, 3)])    # pointwise, large tiles among them; taps
@pytest.mark.parametrize("oc", [208, 200, 196, 198, 195, 129])
@pytest.mark.parametrize("out_dtype", [np.int8, np.int16])
@pytest.mark.parametrize("w_zp", [0, -3])
def test_fused_rescale_rows(ctx, case, oc, out_dtype, w_zp):
    n, hw, ic, k = case
    rng = np.random.default_rng(oc + hw)
    x, w = rng.integers(-128, 128, (n, hw, hw, ic)).astype(np.int8), rng.integers(-128, 128, (oc, k, k, ic)).astype(np.int8)
    bias = rng.integers(-9999, 9999, oc).astype(np.int32)
    mult, shift = rng.integers(1 << 30, 1 << 31, oc).astype(np.int32), rng.integers(37, 43, oc).astype(np.int8)
    out_zp, clamp = (-5, (-100, 110)) if out_dtype == np.int8 else (0, None)
    pad = (k // 2,) * 4
    got, st = gpu_ops.conv2d(ctx, x, w, bias, pad, in_zp=4, w_zp=w_zp, clamp=clamp,
                             rescale=dict(mult=mult, shift=shift, out_zp=out_zp, out_dtype=out_dtype))
    assert ctx.last_kernel.startswith("gemm_mfma_i8_rescale")
    acc = cases.conv2d_exact_blas(x, w, bias, pad, (1, 1), (1, 1), 4, w_zp)
    want, wst = oracle.rescale(acc, mult, shift, out_zp=out_zp, out_dtype=out_dtype)
    assert st == wst == capi.VALID and np.array_equal(got, oracle.clamp(want, *clamp) if clamp else want)
