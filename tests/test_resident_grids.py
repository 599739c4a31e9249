"""Kernels whose workgroups stage their weights and then walk many tiles are launched with as many workgroups as the chip holds at once: one
more would stage its weights only to begin when another ends.  The launcher runs on the CPU on the stand-in of test_lds_grants.py; how many
a CU holds is what the registers of the built kernel leave."""
import functools
import os
import re
import shutil
import subprocess
import sys

import pytest

from reference_model_amd import build
from test_lds_grants import ROOT, RUNTIME

CALL = r"""
import ctypes, sys
i32, vp = ctypes.c_int32, ctypes.c_void_p
fake = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)
lib = ctypes.CDLL(sys.argv[2])
g = (i32 * 17)(*map(int, sys.argv[3].split(",")))
f = getattr(lib, "_ZN3tmi20launch_conv_i16_tapsEP12ihipStream_tRKNS_8ConvGeomEPKvS6_S6_PvS6_b")
f.restype = ctypes.c_char_p
A = vp(1 << 40)    # operands are never touched here
assert f(None, g, A, A, A, A, A, False) == b"conv2d_mfma_i16_i48"
print(fake.last_grid())
"""


@functools.lru_cache(None)
def waves_per_simd(kernel):
    """by the registers the compiler gives every instantiation of a kernel of conv_i16_taps.hip: {(channel tiles, split, ragged): waves}"""
    cmd = [build._hipcc(), *build.HIPCC_FLAGS, "-Rpass-analysis=kernel-resource-usage", "-fno-caret-diagnostics", "--offload-device-only", "-S",
           "-o", os.devnull, os.path.join(build.CSRC, "conv_i16_taps.hip")]
    r = subprocess.run(cmd, capture_output=True, text=True, check=True)
    found, name = {}, ""
    for line in r.stderr.splitlines():
        if "Function Name:" in line:
            m = re.search(kernel + r"ILi(\d)ELb([01])ELb([01])E", line)
            name = (int(m[1]), int(m[2]), int(m[3])) if m else ""
        m = re.search(r"Occupancy \[waves/SIMD\]: (\d+)", line)
        if m and name:
            found[name] = int(m[1])
    return found


# rows of 64 pixels, input and output channels of a 1x1 layer: one block of channels, little LDS, 3072 rounds of four tiles
@pytest.mark.parametrize("rows, ic, oc", [(3072, 20, 16), (3072, 21, 32), (3072, 33, 64), (3072, 16, 16)])
def test_no_more_workgroups_than_the_registers_hold(tmp_path, rows, ic, oc):
    lib = os.path.join(ROOT, "reference_model_amd", "libtosa_mi355.so")
    cc = shutil.which("gcc") or shutil.which("cc")
    if not cc or not os.path.exists(lib):
        pytest.skip("needs a C compiler and the built library")
    src, so = tmp_path / "runtime.c", tmp_path / "runtime.so"
    src.write_text(RUNTIME.replace("int hipLaunchKernel(", "static int grid_x;\nint last_grid(void) { return grid_x; }\nint hipLaunchKernel(")
                   .replace("(void)grid, (void)block", "grid_x = (int)grid.x, (void)block"))
    subprocess.run([cc, "-shared", "-fPIC", "-O1", "-o", str(so), str(src)], check=True)
    geom = (1, rows, 64, ic, oc, 1, 1, rows, 64, 0, 0, 1, 1, 1, 1, oc, 1)
    r = subprocess.run([sys.executable, "-c", CALL, str(so), lib, ",".join(map(str, geom))], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stderr
    ragged = int(ic % 16 != 0)
    held = {w for (_, split, rag), w in waves_per_simd("conv_i16_taps_kernel").items() if rag == ragged and not split}
    assert 2 * 256 < int(r.stdout) <= 256 * min(held)    # (a workgroup is a wave on each SIMD)
