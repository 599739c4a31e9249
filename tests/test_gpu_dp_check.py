"""The DOT_PRODUCT check on its own: sizes from one workgroup to many, fresh results call after call, a check behind work of several
milliseconds, and a stream with nothing left to do when the call returns."""
import ctypes

import numpy as np
import pytest

import dot_product_check as dp
from reference_model_amd import Context, capi

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = Context(0)
    yield c
    c.close()


def _data(rng, n):
    ref = rng.normal(0, 3, n)
    bnd = np.abs(ref) + np.abs(rng.normal(0, 3, n))
    return ref, bnd, (ref + rng.normal(0, 0.7, n) * bnd * 2.0 ** -24).astype(np.float32)


@pytest.mark.parametrize("n", [1, 511, 512, 513, 512 * 32, 512 * 32 + 1, 40_000])
def test_every_call_brings_its_own_results(ctx, n):
    rng = np.random.default_rng(n)
    sets = []
    for i in range(3):
        ref, bnd, imp = _data(rng, n)
        imp[n // 2] += np.float32(1000 * bnd[n // 2] * i)    # the first set passes
        sets.append(([ctx.upload(imp), ctx.upload(ref, capi.F64), ctx.upload(bnd, capi.F64)], dp.check(imp.astype(np.float64), ref, bnd, "fp32", 9)))
    for i in (0, 1, 2, 1, 0, 0, 2):
        r = ctx.dot_product_check(capi.FP32, n, *sets[i][0], 9)
        want = sets[i][1]
        assert r.elements == n and r.failed_elements == (1 if i else 0) and bool(r.compliant) == want["ok"]
        assert r.max_abs_err == pytest.approx(want["max_err"], rel=1e-12) and r.err_sumsq == pytest.approx(want["err_sumsq"], rel=1e-9)


def test_behind_work_of_several_milliseconds(ctx):
    rng = np.random.default_rng(1)
    ref, bnd, imp = _data(rng, 3000)
    dev = [ctx.upload(imp), ctx.upload(ref, capi.F64), ctx.upload(bnd, capi.F64)]
    want = dp.check(imp.astype(np.float64), ref, bnd, "fp32", 9)
    n, hw, c = 4, 56, 128
    d = ctx.conv_desc(capi.FP32, capi.FP32, (n, hw, hw, c), c, 3, 3, (hw, hw), (1, 1, 1, 1), (1, 1), (1, 1), c)
    ops = [ctx.upload(rng.normal(0, 1, s).astype(np.float32)) for s in ((n, hw, hw, c), (c, 3, 3, c), (c,))]
    out = ctx.empty((n, hw, hw, c), capi.F64)
    for _ in range(60):
        ctx.conv2d_precise(d, *ops, False, out)
    r = ctx.dot_product_check(capi.FP32, 3000, *dev, 9)
    assert r.failed_elements == 0 and r.max_abs_err == pytest.approx(want["max_err"], rel=1e-12)
    assert r.err_sumsq == pytest.approx(want["err_sumsq"], rel=1e-9)


@pytest.mark.parametrize("n", [1, 512, 512 * 32, 40_000])
def test_the_stream_is_idle_on_return(n):
    c = Context(0)
    hip = c.lib    # (the runtime the library is linked with)
    stream = ctypes.c_void_p()
    assert hip.hipStreamCreate(ctypes.byref(stream)) == 0
    try:
        c.set_stream(stream.value)
        ref, bnd, imp = _data(np.random.default_rng(n), n)
        dev = [c.upload(imp), c.upload(ref, capi.F64), c.upload(bnd, capi.F64)]
        left = []
        for _ in range(200):
            c.dot_product_check(capi.FP32, n, *dev, 9)
            left.append(hip.hipStreamQuery(stream))
        assert not any(left)
    finally:
        c.close()
        hip.hipStreamDestroy(stream)
