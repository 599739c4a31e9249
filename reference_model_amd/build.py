"""Builds libtosa_mi355.so (HIP kernels + C ABI) for gfx950 with hipcc, in-tree.

    python -m reference_model_amd.build [--force]

hipcc cross-compiles without a GPU.  Every translation unit is compiled to an object file under
csrc/build/ (in parallel) and linked into reference_model_amd/libtosa_mi355.so; the C++ host side (the runner, its
known-answer tests and, where Python's headers are installed, its operator calls as an extension) is built on top of it with g++.
"""
from __future__ import annotations

import concurrent.futures
import os
import re
import shutil
import subprocess
import sys
import sysconfig
import tempfile

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
INCLUDE = os.path.join(os.path.dirname(HERE), "include")
BUILD = os.path.join(CSRC, "build")
LIB = os.path.join(HERE, "libtosa_mi355.so")
HOST_BIN = os.path.join(HERE, "tosa_mi355_run")
CALLS = os.path.join(HERE, "_calls" + sysconfig.get_config_var("EXT_SUFFIX"))    # of this interpreter's ABI: no other loads it

ARCH = "gfx950"
# -packed-fp32-ops off: hipcc must not form v_pk_*_f32 from float code on this hardware pool.
# -ffp-contract=off: the direct floating-point kernels reproduce the reference's separate multiply/add.
HIPCC_FLAGS = [
    "-O3", "-std=c++17", "-fPIC", f"--offload-arch={ARCH}", "-ffp-contract=off",
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wall", "-Wno-unused-function", "-Wno-unknown-cuda-version",
    f"-I{INCLUDE}", f"-I{CSRC}",
]


def _hipcc() -> str:
    exe = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not os.path.exists(exe):
        raise RuntimeError("hipcc not found: cannot build the gfx950 kernels")
    return exe


def sources():
    return sorted(f for f in os.listdir(CSRC) if f.endswith(".hip"))


def kernels_with_scratch(remarks: str) -> list:
    """From the compiler's kernel-resource-usage remarks: "kernel: N bytes per lane" for every kernel whose
    ScratchSize is not zero."""
    kernel, found = "", []
    for line in remarks.splitlines():
        if "Function Name:" in line:
            kernel = line.split("Function Name:")[1].split("[-Rpass")[0].strip()
        elif "ScratchSize [bytes/lane]:" in line:
            size = int(line.split("ScratchSize [bytes/lane]:")[1].split("[-Rpass")[0])
            if size > 0:
                found.append(f"{kernel}: {size} bytes per lane")
    return found


_LISTED = re.compile(r"^<(?P<kernel>[^>\n]+)>:$"
                     r"|^\s*(?P<shift>v_(?:lshlrev_b64|lshrrev_b64|ashrrev_i64))\S*\s+v\[\d+:\d+\],\s*v(?P<amount>\d+),", re.M)


def shifts_by_the_last_register(remarks: str, listing: str) -> list:
    """Kernels in which a 64-bit shift takes its amount from the last vector register of the wave's allocation (registers are
    allocated in blocks of eight), from the compiler's kernel-resource-usage remarks and the objects' disassembly."""
    kernel, registers = "", {}
    for line in remarks.splitlines():
        if "Function Name:" in line:
            kernel = line.split("Function Name:")[1].split("[-Rpass")[0].strip()
        else:
            m = re.search(r"\b(VGPRs|AGPRs): (\d+)", line)
            if m:
                registers.setdefault(kernel, {})[m.group(1)] = int(m.group(2))
    kernel, found = "", []
    for m in _LISTED.finditer(listing):
        if m.group("kernel"):
            kernel = m.group("kernel")
            continue
        used = registers.get(kernel, {})
        # (accumulation registers, where a kernel has any, come behind the others)
        if not used.get("AGPRs") and used.get("VGPRs", 0) % 8 == 0 and int(m.group("amount")) == used.get("VGPRs", 0) - 1:
            entry = f"{kernel}: {m.group('shift')} by v{m.group('amount')} of {used['VGPRs']} registers"
            if entry not in found:
                found.append(entry)
    return found


def _device_listing(obj: str) -> str:
    """The disassembly of the gfx950 code in a freshly compiled object file."""
    tools = os.path.join(os.path.dirname(os.path.dirname(os.path.realpath(_hipcc()))), "llvm", "bin")
    with tempfile.TemporaryDirectory() as tmp:
        fat, code = os.path.join(tmp, "fat"), os.path.join(tmp, "code")
        for cmd in ([os.path.join(tools, "llvm-objcopy"), f"--dump-section=.hip_fatbin={fat}", obj, os.path.join(tmp, "rest.o")],
                    [os.path.join(tools, "clang-offload-bundler"), "--unbundle", "--type=o", f"--targets=hipv4-amdgcn-amd-amdhsa--{ARCH}",
                     f"--input={fat}", f"--output={code}"],
                    [os.path.join(tools, "llvm-objdump"), "-d", "--no-leading-addr", code]):
            r = subprocess.run(cmd, capture_output=True, text=True)
            if r.returncode != 0:
                raise RuntimeError(f"{cmd[0]} failed on {obj}:\n{r.stdout}\n{r.stderr}")
        return r.stdout


def _compile(src: str, force: bool) -> str:
    obj = os.path.join(BUILD, src[:-4] + ".o")
    deps = [os.path.join(CSRC, src)] + [os.path.join(CSRC, h) for h in os.listdir(CSRC) if h.endswith(".h")]
    deps.append(os.path.join(INCLUDE, "tosa_mi355.h"))
    if not force and os.path.exists(obj) and all(os.path.getmtime(obj) >= os.path.getmtime(d) for d in deps):
        return obj
    # -Rpass-analysis=kernel-resource-usage: the compiler reports registers and scratch per kernel.  A kernel with a
    # scratch segment (spilled registers, or a register array indexed at run time) is refused here: on MI355X such
    # kernels were measured 1.5 to 2.5 times slower than the same kernel without one.
    cmd = [_hipcc(), *HIPCC_FLAGS, "-Rpass-analysis=kernel-resource-usage", "-fno-caret-diagnostics", "-c", os.path.join(CSRC, src), "-o", obj]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"hipcc failed on {src}:\n{r.stdout}\n{r.stderr}")
    with_scratch = kernels_with_scratch(r.stderr)
    if with_scratch:
        os.remove(obj)
        raise RuntimeError(f"{src}: kernels with a scratch segment:\n  " + "\n  ".join(with_scratch))
    # A kernel that shifts 64 bits by the last register of its allocation is refused: one such kernel (v87 of 88 registers) shifted
    # by something else now and then, always in the element whose amount lay there, and never with the amount in another
    # register.  Naming a register of the next block of eight in an empty asm moves the border.
    by_last = shifts_by_the_last_register(r.stderr, _device_listing(obj))
    if by_last:
        os.remove(obj)
        raise RuntimeError(f"{src}: 64-bit shifts by the last register of the allocation:\n  " + "\n  ".join(by_last))
    warn = "\n".join(l for l in r.stderr.splitlines()
                     if "packed-fp32-ops" not in l and "-Rpass-analysis" not in l and l.strip())
    if warn:
        sys.stderr.write(warn + "\n")
    return obj


def build(force: bool = False, jobs: int = 8) -> str:
    os.makedirs(BUILD, exist_ok=True)
    srcs = sources()
    with concurrent.futures.ThreadPoolExecutor(max_workers=min(jobs, len(srcs))) as ex:
        objs = list(ex.map(lambda s: _compile(s, force), srcs))
    if force or not os.path.exists(LIB) or any(os.path.getmtime(o) > os.path.getmtime(LIB) for o in objs):
        cmd = [_hipcc(), "-shared", "-fPIC", f"--offload-arch={ARCH}", "-o", LIB, *objs]
        r = subprocess.run(cmd, capture_output=True, text=True)
        if r.returncode != 0:
            raise RuntimeError(f"link failed:\n{r.stdout}\n{r.stderr}")
    return LIB


def build_host(force: bool = False) -> list:
    """Compiles the C++ host side above the C ABI (g++, links against libtosa_mi355.so):
    tosa_mi355_run (command-line runner) and tosa_mi355_host_kats (known-answer tests)."""
    host = os.path.join(CSRC, "host")
    common = [os.path.join(host, f) for f in ("formats.cc", "runtime.cc")]
    outs = []
    for exe, main in ((HOST_BIN, "main.cc"), (os.path.join(HERE, "tosa_mi355_host_kats"), "host_kats.cc")):
        srcs = common + [os.path.join(host, main)]
        deps = srcs + [os.path.join(host, "tosa_host.h"), os.path.join(INCLUDE, "tosa_mi355.h"), LIB]
        if force or not os.path.exists(exe) or any(os.path.getmtime(d) > os.path.getmtime(exe) for d in deps):
            cmd = ["g++", "-O2", "-std=c++17", "-Wall", "-Wextra", f"-I{INCLUDE}", f"-I{host}", *srcs, "-o", exe,
                   f"-L{HERE}", "-ltosa_mi355", "-Wl,-rpath,$ORIGIN", "-Wl,-rpath-link," + "/opt/rocm/lib"]
            r = subprocess.run(cmd, capture_output=True, text=True)
            if r.returncode != 0:
                raise RuntimeError(f"g++ failed on {main}:\n{r.stdout}\n{r.stderr}")
            if r.stderr.strip():
                sys.stderr.write(r.stderr)
        outs.append(exe)
    calls = build_calls(force)
    return outs + [calls] if calls else outs


def build_calls(force: bool = False) -> str | None:
    """The operator calls of capi.Context as a CPython extension; None where Python's headers are not installed (the calls then
    stay on ctypes)."""
    src, headers = os.path.join(CSRC, "host", "pycalls.cc"), sysconfig.get_paths()["include"]
    untagged = os.path.join(HERE, "_calls.so")    # what an interpreter of any version would load
    if os.path.exists(untagged):
        os.remove(untagged)
    if not os.path.exists(os.path.join(headers, "Python.h")):
        sys.stderr.write(f"no Python.h under {headers}: the operator calls stay on ctypes\n")
        return None
    if force or not os.path.exists(CALLS) or any(os.path.getmtime(d) > os.path.getmtime(CALLS) for d in (src, os.path.join(INCLUDE, "tosa_mi355.h"))):
        cmd = ["g++", "-O2", "-std=c++17", "-Wall", "-Wextra", "-Wno-missing-field-initializers", "-fPIC", "-shared", f"-I{INCLUDE}",
               f"-I{headers}", src, "-o", CALLS, f"-L{HERE}", "-ltosa_mi355", "-Wl,-rpath,$ORIGIN", "-Wl,-rpath-link,/opt/rocm/lib"]
        r = subprocess.run(cmd, capture_output=True, text=True)
        if r.returncode != 0:
            raise RuntimeError(f"g++ failed on pycalls.cc:\n{r.stdout}\n{r.stderr}")
        if r.stderr.strip():
            sys.stderr.write(r.stderr)
    return CALLS


if __name__ == "__main__":
    print(build(force="--force" in sys.argv))
    print(build_host(force="--force" in sys.argv))
