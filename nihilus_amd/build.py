"""Builds libnihilus_q8_hip.so (the gfx950 Q8_0 kernels + their C ABI) in-tree with hipcc."""
from __future__ import annotations

import os
import shutil
import subprocess
import sys
import sysconfig
from concurrent.futures import ThreadPoolExecutor

PKG_DIR = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(PKG_DIR, "csrc")
OBJ_DIR = os.path.join(CSRC, "build")
LIB_NAME = "libnihilus_q8_hip.so"
LIB_PATH = os.path.join(PKG_DIR, LIB_NAME)

SOURCES = ["q8_0_abi.hip", "q8_0_quantize.hip", "q8_0_layout.hip", "q8_0_get_rows.hip", "q8_0_gemv.hip", "q8_0_gemv_rows.hip", "q8_0_gemv_rows_mfma.hip", "q8_0_gemv_group.hip", "q8_0_mul_mat_f32act.hip", "q8_0_ffn.hip", "q8_0_decode_layer.hip", "q8_0_gemm.hip", "q8_0_gemm_skinny.hip", "q8_0_gemm_rows.hip", "q8_0_profile.hip", "gguf_q8_0.cpp"]

# -packed-fp32-ops off: v_pk_{add,mul,fma}_f32 are kept out of the generated code on purpose.
# No -ffast-math: the quantizer needs IEEE divide, unfused multiply and round-half-even.
HIPCC_FLAGS = [
    "--offload-arch=gfx950",
    "-O3",
    "-std=c++20",
    "-fPIC",
    "-fno-fast-math",
    "-ffp-contract=off",
    "-Wall",
    "-Wextra",
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    # MFMA results stay in ordinary VGPRs: the mat-mat converts every int32 block sum on the VALU right away, and a
    # result parked in an accumulation register would cost one extra copy instruction per value (doubling the VALU work)
    "-mllvm", "-amdgpu-mfma-vgpr-form",
]
# A kernel's first arguments (up to sixteen dwords) arrive in scalar registers with the wave instead of being read from memory by it, a miss of the scalar
# cache in front of the first address; kernels name what that address takes first.  norm + quantize of 4 rows 3.14 -> 2.95 us, of 16 3.48 -> 3.33, of [64 x 8192]
# 4.38 -> 4.14; mul_mat of 2 to 16 rows, 60 random shapes of each number, 1.03 to 1.05 times as fast.
PRELOAD_FLAGS = ["-mllvm", "-amdgpu-kernarg-preload-count=16"]
# not where a launch is many short waves, each of which then starts later: embedding rows of 4 tokens 1.83 us without, 1.99 with; [14336 x 4096] into the
# device layout 25.0 / 25.8
NO_PRELOAD = ("q8_0_get_rows.hip", "q8_0_layout.hip")
# The wrappers' native calls, a CPython module against torch's own headers and libraries (which are loaded with torch, before it).  Not part of
# the library, whose other users need no torch, and the wrappers work without it.
CALLS_SOURCE = "py_calls.cpp"
CALLS_PATH = os.path.join(PKG_DIR, "_calls" + sysconfig.get_config_var("EXT_SUFFIX"))
# the host pass does not know the packed-fp32 feature name and says so once per source: not an error
NOISE = "is not a recognized feature for this target"


def hipcc() -> str:
    exe = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not os.path.exists(exe):
        raise RuntimeError("hipcc not found; the Q8_0 library can only be built with ROCm's hipcc")
    return exe


def _run(cmd: list[str]) -> str:
    res = subprocess.run(cmd, capture_output=True, text=True)
    err = "\n".join(l for l in res.stderr.splitlines() if NOISE not in l)
    if res.returncode != 0:
        raise RuntimeError(f"hipcc failed ({res.returncode}):\n{' '.join(cmd)}\n{err}")
    return err


def _newest_header_mtime(include: str) -> float:
    newest = 0.0
    for folder in (CSRC, os.path.join(include, "nihilus_amd")):
        for name in os.listdir(folder):
            if name.endswith(".h"):
                newest = max(newest, os.path.getmtime(os.path.join(folder, name)))
    return newest


def build_library(verbose: bool = False, extra_flags: list[str] | None = None, incremental: bool = False, jobs: int = 8) -> str:
    """Compile every HIP source to an object (in parallel) and link them into one shared library next to this file.

    Recompiles everything unless incremental=True, which keeps objects newer than their source and every header.
    """
    include = os.path.join(os.path.dirname(PKG_DIR), "include")
    os.makedirs(OBJ_DIR, exist_ok=True)
    flags = [*HIPCC_FLAGS, "-I", include, *(extra_flags or [])]
    headers = _newest_header_mtime(include)

    def compile_one(src: str) -> str:
        path = os.path.join(CSRC, src)
        obj = os.path.join(OBJ_DIR, os.path.splitext(src)[0] + ".o")
        preload = PRELOAD_FLAGS if src.endswith(".hip") and src not in NO_PRELOAD else []
        if incremental and not extra_flags and os.path.exists(obj) and os.path.getmtime(obj) > max(os.path.getmtime(path), headers):
            return ""
        return _run([hipcc(), *flags, *preload, "-c", path, "-o", obj])

    with ThreadPoolExecutor(max_workers=max(1, jobs)) as pool:
        notes = list(pool.map(compile_one, SOURCES))
    objs = [os.path.join(OBJ_DIR, os.path.splitext(s)[0] + ".o") for s in SOURCES]
    notes.append(_run([hipcc(), "--offload-arch=gfx950", "-shared", "-fPIC", "-o", LIB_PATH, *objs]))
    if verbose:
        text = "\n".join(n for n in notes if n.strip())
        if text:
            print(text)
    return LIB_PATH


def calls_tag() -> str:
    """What the module of the native calls is built for: it reads torch's and CPython's structures by their layout, so by no other one."""
    import torch

    return f"torch {torch.__version__} {sys.implementation.cache_tag}"


def build_calls(incremental: bool = False) -> str:
    """Compile the CPython module behind the wrappers of nihilus_amd/q8_0.py (host code only), linked against the library beside it."""
    tag = calls_tag()
    import torch

    include = os.path.join(os.path.dirname(PKG_DIR), "include")
    path = os.path.join(CSRC, CALLS_SOURCE)
    if incremental and os.path.exists(CALLS_PATH) and os.path.getmtime(CALLS_PATH) > max(os.path.getmtime(path), _newest_header_mtime(include)):
        with open(CALLS_PATH, "rb") as f:
            if tag.encode() + b"\0" in f.read():
                return ""
    os.makedirs(OBJ_DIR, exist_ok=True)
    root = os.path.dirname(torch.__file__)
    rocm = os.path.dirname(os.path.dirname(os.path.realpath(hipcc())))
    system = [os.path.join(rocm, "include"), os.path.join(root, "include"), os.path.join(root, "include", "torch", "csrc", "api", "include"), sysconfig.get_paths()["include"]]
    obj = os.path.join(OBJ_DIR, "py_calls.o")
    note = _run([hipcc(), "-x", "c++", "-O2", "-std=c++20", "-fPIC", "-Wall", "-Wextra", "-DUSE_ROCM=1", "-D__HIP_PLATFORM_AMD__=1", f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}",
                 f'-DNH_BUILT_FOR="{tag}"', "-I", include, *(x for d in system for x in ("-isystem", d)), "-c", path, "-o", obj])
    return note + _run([hipcc(), "-shared", "-fPIC", "-o", CALLS_PATH, obj, "-L", os.path.join(root, "lib"), "-L", PKG_DIR, "-ltorch_python", "-ltorch_cpu", "-lc10", "-lc10_hip", f"-l:{LIB_NAME}",
                        "-Wl,-rpath,$ORIGIN"])


if __name__ == "__main__":
    print(build_library(verbose=True, incremental="--incremental" in sys.argv))
    try:
        print(build_calls("--incremental" in sys.argv) or CALLS_PATH)
    except Exception as e:  # noqa: BLE001 -- no torch, or headers that do not fit: the library is whole, the wrappers take the Python way
        print(f"the wrappers' native calls were not built: {e}", file=sys.stderr)
