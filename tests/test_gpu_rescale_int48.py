"""RESCALE of INT48 with 16-bit multipliers on the kernel that walks down the rows: against the oracle, at its edges, where a value needs its 48th
bit extended, and with what raises flags: shifts and multipliers out of range, results past 32 bits."""
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


@pytest.mark.parametrize("rows, c", [(75001, 4), (3001, 100), (4700, 64), (294, 1024), (40000, 8)])
@pytest.mark.parametrize("out", [np.int8, np.int16, np.int32])
@pytest.mark.parametrize("kind", ["plain", "uniform", "large", "negative", "shift"])
def test_int48(ctx, rows, c, out, kind):
    rng = np.random.default_rng(rows + c)
    x = rng.integers(-(1 << 40), 1 << 40, (rows, c), dtype=np.int64)
    x.flat[:4] = [-(1 << 47), (1 << 47) - 1, 0, -1]
    n = 1 if kind == "uniform" else c
    mult, shift = rng.integers(1 << 14, 1 << 15, n).astype(np.int16), rng.integers(38, 46, n).astype(np.int8)
    if kind == "large":
        shift[0] = 20    # results of more than 32 bits
    if kind == "negative":
        mult[n // 2] = -5
    if kind == "shift":
        shift[n // 2] = 1
    zp = 3 if out == np.int8 else 0
    args = dict(out_zp=3 if out == np.int8 else 0, out_dtype=out, scale32=False, rounding_mode=capi.ROUND_SINGLE, per_channel=n > 1)
    got, st = gpu_ops.rescale(ctx, x, mult, shift, **args)
    assert ctx.last_kernel == "rescale_i48"
    want, wst = oracle.rescale(x, mult, shift, **args)
    assert st == wst and (st == capi.VALID) == (kind in ("plain", "uniform"))
    if st != capi.VALID:    # (the oracle has no values then: the general kernel's, on pieces that are left to it)
        want = np.concatenate([gpu_ops.rescale(ctx, part, mult, shift, **args)[0] for part in np.array_split(x, 4)])
    assert np.array_equal(got, want)
