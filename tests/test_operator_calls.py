"""The two forms of the binding's operator calls, ctypes and native: the same names, arguments, results and errors (no GPU needed: a
context that does not exist refuses every call with the library's own message)."""
import ctypes
import inspect
import subprocess
import sys

import pytest

from reference_model_amd import TmiError, build, capi

capi.load_library()
NATIVE = {name: vars(capi.Context)[name] for name in capi.PLAIN_OPERATORS}
CONV = (capi.ConvDesc(), 0, 0, 0, 0, 0)
FUSED = CONV + (capi.RescaleDesc(), 0, 0, 0)
CALLS = {"conv2d": CONV + (0,), "depthwise_conv2d": CONV + (0,), "transpose_conv2d": (capi.TconvDesc(),) + CONV[1:] + (0,),
         "conv3d": (capi.Conv3dDesc(),) + CONV[1:] + (0,), "conv2d_rescale_clamp": FUSED, "depthwise_conv2d_rescale_clamp": FUSED,
         "matmul": (capi.INT8, 1, 1, 1, 1, 0, 0, 0, 0, 0), "rescale": (capi.RescaleDesc(), 1, 1, 1, 0, 0, 0, 0),
         "clamp": (capi.INT8, 1, 0, 0, 0, 0), "avg_pool2d": (capi.PoolDesc(), 0, 0, 0, 0), "max_pool2d": (capi.PoolDesc(), 0, 0)}


@pytest.fixture
def nothing():
    """a Context whose library is loaded and whose handle is none"""
    c = object.__new__(capi.Context)
    c.lib, c.handle = capi.load_library(), None
    return c


def test_native_calls_are_the_ones_in_use():
    assert set(NATIVE) == set(CALLS) and all(NATIVE[n] is not capi.PLAIN_OPERATORS[n] for n in NATIVE)
    for name, plain in capi.PLAIN_OPERATORS.items():
        assert list(inspect.signature(NATIVE[name]).parameters) == list(inspect.signature(plain).parameters)


@pytest.mark.parametrize("form", ["native", "plain"])
@pytest.mark.parametrize("name", list(CALLS))
def test_arguments_and_errors_of_both_forms(nothing, form, name):
    fn, args = (NATIVE if form == "native" else capi.PLAIN_OPERATORS)[name], CALLS[name]
    call = lambda *a, **k: fn.__get__(nothing, capi.Context)(*a, **k)  # noqa: E731
    with pytest.raises(TmiError) as e:
        call(*args)
    assert e.value.status == capi.ERROR and "null context" in e.value.message
    names = list(inspect.signature(capi.PLAIN_OPERATORS[name]).parameters)[1:]
    with pytest.raises(TmiError):
        call(**dict(zip(names, args)))
    if name.endswith("clamp") and name != "clamp":
        with pytest.raises(TmiError):
            call(*args, clamp=(-5, 5))
        with pytest.raises(ValueError):
            call(*args, clamp=(-5, 5, 6))
    with pytest.raises(TypeError):
        call(*args[:-1])
    with pytest.raises(TypeError):
        call(*args, no_such_argument=1)
    with pytest.raises((TypeError, ctypes.ArgumentError)):
        call(*args[:-1], "no tensor")


def test_the_binding_works_without_the_extension():
    """another interpreter, or a build without Python's headers: every operator on ctypes"""
    code = ("import sys; sys.modules['reference_model_amd._calls'] = None\n"
            "from reference_model_amd import capi\n"
            "assert all(hasattr(capi.Context, n) for n in capi.PLAIN_OPERATORS)\n"
            "capi.load_library()\n"
            "assert all(vars(capi.Context)[n] is f for n, f in capi.PLAIN_OPERATORS.items())\n")
    r = subprocess.run([sys.executable, "-c", code], capture_output=True, text=True, cwd=build.HERE + "/..")
    assert r.returncode == 0, r.stderr


def test_the_build_goes_on_without_pythons_headers(monkeypatch, tmp_path):
    monkeypatch.setattr(build.sysconfig, "get_paths", lambda: {"include": str(tmp_path)})
    assert build.build_calls() is None
