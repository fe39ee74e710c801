"""Builds libvoxattn.so in-tree with hipcc for gfx950 (run as ``python -m voxcpm2_arabic_dialects_turbo_amd.build``).

The attention library is one shared library, C ABI only (include/vox_attn.h): no torch headers, no pybind. The
sources compile in parallel and link into ``voxcpm2_arabic_dialects_turbo_amd/libvoxattn.so``. Beside it, ``_calls`` is
the CPython module through which the operators call it (csrc/host_calls.cpp, host code only; without Python's headers it
is left out and the same entry points are called through ctypes), and
``libvoxprobe.so`` (include/vox_probe.h) holds the memory-rate probes bench.py runs; the attention path never loads
it. Packed FP32 VALU instructions are disabled for
device code (``-packed-fp32-ops``); hipcc's host pass warns that it does not know that feature, which is harmless.
"""

from __future__ import annotations

import os
import shutil
import subprocess
import sys
import sysconfig
from concurrent.futures import ThreadPoolExecutor

PKG_DIR = os.path.dirname(os.path.abspath(__file__))
REPO_DIR = os.path.dirname(PKG_DIR)
CSRC = os.path.join(PKG_DIR, "csrc")
BUILD_DIR = os.path.join(PKG_DIR, "_build")
LIB_NAME = "libvoxattn.so"
LIB_PATH = os.path.join(PKG_DIR, LIB_NAME)
SOURCES = ["store_kvcache.hip", "decode_attn.hip", "prefill_attn.hip", "quantize_rows.hip", "kv_copy.hip", "capi.hip"]
PROBE_PATH = os.path.join(PKG_DIR, "libvoxprobe.so")
PROBE_SOURCES = ["bench_probe.hip"]
# the CPython entry to the C ABI (host code only), for the interpreter that builds it
CALLS_PATH = os.path.join(PKG_DIR, "_calls" + (sysconfig.get_config_var("EXT_SUFFIX") or ".so"))
CALLS_SOURCE = "host_calls.cpp"
ARCH = "gfx950"


def hipcc() -> str:
    for cand in (os.environ.get("HIPCC"), shutil.which("hipcc"), "/opt/rocm/bin/hipcc"):
        if cand and os.path.exists(cand):
            return cand
    raise RuntimeError("hipcc not found: the HIP toolchain (ROCm) is required to build libvoxattn.so")


def compile_flags() -> list[str]:
    return [
        f"--offload-arch={ARCH}",
        "-O3",
        "-std=c++17",
        "-fPIC",
        "-munsafe-fp-atomics",
        "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
        f"-I{os.path.join(REPO_DIR, 'include')}",
        f"-I{CSRC}",
    ]


def _run(cmd: list[str]) -> None:
    proc = subprocess.run(cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
    # the host pass's "not a recognized feature" warnings for -packed-fp32-ops are expected noise
    noise = "'-packed-fp32-ops' is not a recognized feature"
    text = "\n".join(line for line in proc.stdout.splitlines() if noise not in line)
    if proc.returncode != 0:
        raise RuntimeError(f"command failed ({proc.returncode}): {' '.join(cmd)}\n{text}")
    if text.strip():
        print(text, file=sys.stderr)


def _python_include() -> str | None:
    """The directory of Python.h, None where Python's headers are not installed."""
    path = sysconfig.get_paths()["include"]
    return path if os.path.exists(os.path.join(path, "Python.h")) else None


def build(verbose: bool = False) -> str:
    """Compiles every source and links libvoxattn.so and libvoxprobe.so and the CPython module; returns the attention
    library's path. Always rebuilds; what was built before is replaced only when everything compiles, all of it."""
    cc = hipcc()
    os.makedirs(BUILD_DIR, exist_ok=True)
    cmds = []
    for src in SOURCES + PROBE_SOURCES:
        obj = os.path.join(BUILD_DIR, src.replace(".hip", ".o"))
        cmds.append([cc, *compile_flags(), "-c", os.path.join(CSRC, src), "-o", obj])
    include = _python_include()
    built = [LIB_PATH, PROBE_PATH]
    if include is not None:
        cxx = os.environ.get("CXX") or shutil.which("g++") or cc
        cmds.append([cxx, "-O2", "-std=c++17", "-shared", "-fPIC", "-fvisibility=hidden", f"-I{include}",
                     os.path.join(CSRC, CALLS_SOURCE), "-o", CALLS_PATH + ".tmp"])
        built.append(CALLS_PATH)
    else:
        print("Python.h not found: the operators will call the library through ctypes", file=sys.stderr)
    with ThreadPoolExecutor(max_workers=min(len(cmds), os.cpu_count() or 1)) as ex:
        for cmd, fut in zip(cmds, [ex.submit(_run, c) for c in cmds]):
            if verbose:
                print(" ".join(cmd))
            fut.result()
    for path, srcs in ((LIB_PATH, SOURCES), (PROBE_PATH, PROBE_SOURCES)):
        objs = [os.path.join(BUILD_DIR, src.replace(".hip", ".o")) for src in srcs]
        _run([cc, f"--offload-arch={ARCH}", "-shared", "-fPIC", *objs, "-o", path + ".tmp"])
    for old in (CALLS_PATH, os.path.join(PKG_DIR, "_calls.so")):  # (a module of another build is not left beside these)
        if old not in built and os.path.exists(old):
            os.remove(old)
    for path in built:
        os.replace(path + ".tmp", path)
    return LIB_PATH


if __name__ == "__main__":
    print(build(verbose="-v" in sys.argv))
