"""Launches that ask for more than 64 KB of dynamic LDS: the kernel's own limit is raised first, also where kernels of one signature
are launched one after the other.  The launchers run on the CPU, in a process of their own, on a stand-in for the five runtime calls they
make, which keeps each kernel's limit and what it is launched with."""
import os
import shutil
import subprocess
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

RUNTIME = r"""
#include <stddef.h>
typedef struct { unsigned x, y, z; } dim3;
static const void* kernels[64];
static size_t limits[64];
static int known, launches, beyond;
static int find(const void* k)
{
    for (int i = 0; i < known; i++)
        if (kernels[i] == k)
            return i;
    kernels[known] = k, limits[known] = 65536;
    return known++;
}
int hipGetDevice(int* d) { *d = 0; return 0; }
int hipGetLastError(void) { return 0; }
int hipFuncSetAttribute(const void* k, int attribute, int bytes) { (void)attribute; limits[find(k)] = (size_t)bytes; return 0; }
static dim3 grid_, block_;
static size_t lds_;
static void* stream_;
int __hipPushCallConfiguration(dim3 grid, dim3 block, size_t lds, void* stream) { grid_ = grid, block_ = block, lds_ = lds, stream_ = stream; return 0; }
int __hipPopCallConfiguration(dim3* grid, dim3* block, size_t* lds, void** stream) { *grid = grid_, *block = block_, *lds = lds_, *stream = stream_; return 0; }
int hipLaunchKernel(const void* k, dim3 grid, dim3 block, void** args, size_t lds, void* stream)
{
    (void)grid, (void)block, (void)args, (void)stream;
    launches++, beyond += lds > limits[find(k)];
    return 0;
}
int counts(int* different) { *different = known; return launches * 1000 + beyond; }
"""

CALLS = r"""
import ctypes, sys
i32, i64, vp = ctypes.c_int32, ctypes.c_int64, ctypes.c_void_p
fake = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)    # found before the runtime the library is linked with
lib = ctypes.CDLL(sys.argv[2])
A = vp(1 << 40)    # operands are never touched here
def matmul(in_dtype, n, h, c, w):
    f = getattr(lib, "_ZN3tmi20launch_matmul_raggedEP12ihipStream_tiiiiiPKvS3_iiPv")
    f.restype = ctypes.c_char_p
    assert f(None, in_dtype, n, h, c, w, A, A, 0, 0, A) == b"matmul_ragged_f16"
class Geom(ctypes.Structure):
    _fields_ = [(k, i32) for k in "N IH IW IC OC KH KW OH OW pad_top pad_left stride_y stride_x dil_y dil_x bias_len M".split()]
class Rescale(ctypes.Structure):
    _fields_ = [("multiplier", vp), ("shift", vp)] + [(k, i32) for k in "in_zp out_zp qmin qmax clamp_min clamp_max".split()] + \
        [(k, ctypes.c_uint8) for k in "scale32 double_round inexact_round per_channel in_bits in_unsigned has_clamp enabled fast".split()] + \
        [("lo", i32), ("hi", i32)]
def slab(zp, n):
    g = Geom(n, 56, 56, 64, 64, 3, 3, 56, 56, 1, 1, 1, 1, 1, 1, 64, 1)
    r = Rescale(A, A, 0, 0, -128, 127, 0, 0, 1, 1, 0, 1, 32, 0, 0, 1, 1, -128, 127)
    f = getattr(lib, SLAB)
    f.restype = ctypes.c_char_p
    name = f(None, CODES["int8"], CODES["int8"], ctypes.byref(g), A, A, A, zp, 0, ctypes.byref(r), A, A, A, None, None)
    assert name == b"conv2d_slab_wreg_i8_rescale", name
sys.path.insert(0, sys.argv[3])
from reference_model_amd import capi
CODES = dict(int8=capi.INT8, fp16=capi.FP16)
SLAB = sys.argv[4]
if sys.argv[5] == "matmul":
    matmul(CODES["fp16"], 120, 1, 33 << 20, 1)    # rows of 66 MB, K split over sixteen waves, 128 KB
    matmul(CODES["fp16"], 120, 1, 1 << 20, 1)     # shorter rows of the same form
else:
    for n in (8, 64):    # weights loaded into LDS, through registers
        slab(0, n), slab(5, n)
different = i32()
n = fake.counts(ctypes.byref(different))
print(n // 1000, n % 1000, different.value)
"""


@pytest.mark.parametrize("which, kernels", [("matmul", 2), ("slab", 4)])
def test_every_kernel_has_a_limit_of_its_own(tmp_path, which, kernels):
    lib = os.path.join(ROOT, "reference_model_amd", "libtosa_mi355.so")
    cc = shutil.which("gcc") or shutil.which("cc")
    if not cc or not os.path.exists(lib):
        pytest.skip("needs a C compiler and the built library")
    src, so = tmp_path / "runtime.c", tmp_path / "runtime.so"
    src.write_text(RUNTIME)
    subprocess.run([cc, "-shared", "-fPIC", "-O1", "-o", str(so), str(src)], check=True)
    names = subprocess.run(["nm", "-D", "--defined-only", lib], capture_output=True, text=True, check=True).stdout.split()
    slab = [n for n in names if n.startswith("_ZN3tmi18launch_conv2d_slabE")]
    r = subprocess.run([sys.executable, "-c", CALLS, str(so), lib, ROOT, slab[0], which], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stderr
    launches, beyond, different = map(int, r.stdout.split())
    assert launches == different == kernels and beyond == 0
