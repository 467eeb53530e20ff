"""Builds librlk_hip.so (the C-ABI library of HIP kernels) in-tree for gfx950 with hipcc."""

from __future__ import annotations

import os
import re
import shutil
import subprocess
import sys

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
LIB_DIR = os.path.join(HERE, "lib")
LIB_PATH = os.path.join(LIB_DIR, "librlk_hip.so")

SOURCES = ["rlk_core.hip", "rlk_linear_logp.hip", "rlk_logp_scan.hip", "rlk_grpo.hip",
           "rlk_wide.hip", "rlk_rmsnorm.hip"]

# Packed-fp32 VALU forms are switched off for every device function of this library (the host pass
# of hipcc warns that it does not know the feature; build() checks the device code instead).
HIPCC_FLAGS = [
    "--offload-arch=gfx950", "-O3", "-std=c++17", "-fPIC",
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wall", "-Wno-unused-function",
]


def hipcc() -> str:
    exe = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not os.path.exists(exe):
        raise RuntimeError("hipcc not found; librlk_hip.so cannot be built")
    return exe


def _check_no_packed_fp32(asm_path: str, src: str) -> None:
    """The switch-off of the packed-fp32 VALU forms is a device-side target feature; the host pass
    of hipcc does not know it and says so.  What counts is the device code: it must not contain
    a packed fp32 add / mul / fma."""
    bad = re.compile(r"\bv_pk_(add|mul|fma)_f32\b")
    with open(asm_path) as fh:
        hits = [line.strip() for line in fh if bad.search(line)]
    if hits:
        raise RuntimeError(f"{src}: device code contains packed fp32 instructions "
                           f"({len(hits)}, first: {hits[0]}); the -packed-fp32-ops switch did not take effect")


# Wait states that the hardware wants around a 16-byte store and that the compiler only provides for its own:
# before a matrix instruction's result is stored, and before the stored registers are overwritten.
STREAM_STORE = re.compile(r"global_store_dwordx4 v\[\d+:\d+\], ([av])\[(\d+):(\d+)\], off sc1 nt$")
MFMA_TO_STORE = 12
STORE_TO_WRITE = 2


def _check_stream_stores(asm_path: str, src: str) -> int:
    """The inline-assembly stores (stream_store) are opaque to the compiler's hazard pass: each has to be
    followed by ``s_nop 1`` (or more) at once, and no matrix instruction may write its data within the
    twelve wait states in front of it.  Returns how many there are."""
    with open(asm_path) as fh:
        lines = [line.split(";")[0].strip() for line in fh]
    code = [line for line in lines if line and not line.startswith((".", "//"))]

    def states(line):
        return int(line.split()[1]) + 1 if line.startswith("s_nop") else 1

    found = 0
    for at, line in enumerate(code):
        hit = STREAM_STORE.match(line)
        if hit is None:
            continue
        found += 1
        after = code[at + 1] if at + 1 < len(code) else ""
        if not after.startswith("s_nop") or states(after) < STORE_TO_WRITE:
            raise RuntimeError(f"{src}: '{line}' is followed by '{after}', not by s_nop 1")
        kind, lo, hi = hit.group(1), int(hit.group(2)), int(hit.group(3))
        passed = 0
        for back in range(at - 1, -1, -1):
            if passed >= MFMA_TO_STORE or code[back].endswith(":"):
                break
            wrote = re.match(r"v_mfma\S+ ([av])\[(\d+):(\d+)\]", code[back])
            if wrote and wrote.group(1) == kind and int(wrote.group(2)) <= hi and int(wrote.group(3)) >= lo:
                raise RuntimeError(f"{src}: '{line}' stores the result of '{code[back]}' after {passed} wait states")
            passed += states(code[back])
    return found


def _check_m0_loads(asm_path: str, src: str) -> int:
    """A load to LDS takes its destination from M0, and one wait state has to lie between a scalar write of M0
    and the load; in inline assembly nothing provides it.  Returns how many such loads there are."""
    with open(asm_path) as fh:
        lines = [line.split(";")[0].strip() for line in fh]
    code = [line for line in lines if line and not line.startswith((".", "//"))]
    found = 0
    for before, line in zip([""] + code, code):
        if re.match(r"(global|buffer|scratch)_load_(lds_|\S+.*\blds\b)", line):
            found += 1
            if re.match(r"s_\S+ m0,", before):
                raise RuntimeError(f"{src}: '{line}' follows '{before}' without a wait state")
    return found


def _check_cached_stores(asm_path: str, src: str) -> int:
    """The unchained dW kernel is up to half as slow again with stores past the L2: none of its stores may be one.
    Returns how many such kernels there are."""
    found, inside = 0, None
    with open(asm_path) as fh:
        for line in fh:
            code = line.split(";")[0].strip()
            if re.match(r"\w*linear_logp_dw_kernel\w*:$", code):
                found, inside = found + 1, code
            elif code.startswith("s_endpgm"):
                inside = None
            elif inside and STREAM_STORE.match(code):
                raise RuntimeError(f"{src}: '{code}' in {inside}")
    return found


BINDING_SRC = "rlk_torch_binding.cpp"
BINDING_NAME = "_rlk_C"
BINDING_PATH = os.path.join(LIB_DIR, BINDING_NAME + ".so")


def _binding_compile_cmd(obj: str):
    """hipcc line that compiles the PyTorch binding (host code, torch + pybind11 headers)."""
    import sysconfig

    import torch
    from torch.utils import cpp_extension as ce

    incs = [os.path.join(os.path.dirname(HERE), "include"), *ce.include_paths("cuda"),
            sysconfig.get_paths()["include"]]
    abi = int(bool(getattr(torch._C, "_GLIBCXX_USE_CXX11_ABI", True)))
    return [hipcc(), "--offload-arch=gfx950", "-O2", "-std=c++17", "-fPIC", "-x", "hip", "-c",
            os.path.join(CSRC, BINDING_SRC), "-o", obj, f"-DTORCH_EXTENSION_NAME={BINDING_NAME}",
            "-D__HIP_PLATFORM_AMD__=1", "-DUSE_ROCM=1", "-DTORCH_API_INCLUDE_EXTENSION_H",
            f"-D_GLIBCXX_USE_CXX11_ABI={abi}", "-Wno-unused-result", *[f"-I{i}" for i in incs]]


def _binding_link_cmd(obj: str, out: str):
    from torch.utils import cpp_extension as ce

    torch_lib = ce.library_paths()[0]
    return [hipcc(), "--offload-arch=gfx950", "-shared", "-fPIC", obj, "-o", out, f"-L{torch_lib}",
            "-lc10", "-lc10_hip", "-ltorch_cpu", "-ltorch_hip", "-ltorch", "-ltorch_python",
            f"-L{LIB_DIR}", "-lrlk_hip", "-Wl,-rpath,$ORIGIN", f"-Wl,-rpath,{torch_lib}"]


def build(verbose: bool = False, extra_flags=()) -> str:
    """Compile every source and link the shared library. Always recompiles.  Every source is
    also compiled to device assembly once more to verify that no packed-fp32 instruction was
    generated."""
    os.makedirs(LIB_DIR, exist_ok=True)
    objs = []
    procs = []
    for src in SOURCES:
        path = os.path.join(CSRC, src)
        if not os.path.exists(path):
            raise RuntimeError(f"source file {path} is missing")
        obj = os.path.join(LIB_DIR, src.replace(".hip", ".o"))
        asm = os.path.join(LIB_DIR, src.replace(".hip", ".device.s"))
        cmd = [hipcc(), *HIPCC_FLAGS, *extra_flags, "-c", path, "-o", obj]
        chk = [hipcc(), *HIPCC_FLAGS, *extra_flags, "--cuda-device-only", "-S", path, "-o", asm]
        if verbose:
            print(" ".join(cmd), flush=True)
        procs.append((src, None, subprocess.Popen(cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT)))
        procs.append((src, asm, subprocess.Popen(chk, stdout=subprocess.PIPE, stderr=subprocess.STDOUT)))
        objs.append(obj)
    # the compiled PyTorch binding (the reference's `_C` symbol names over this C ABI): its
    # compile runs beside the kernels', its link needs the library
    bind_obj = os.path.join(LIB_DIR, BINDING_NAME + ".o")
    bind_proc = subprocess.Popen(_binding_compile_cmd(bind_obj), stdout=subprocess.PIPE,
                                 stderr=subprocess.STDOUT)
    for src, asm, proc in procs:
        out = proc.communicate()[0].decode()
        if proc.returncode != 0:
            raise RuntimeError(f"hipcc failed on {src}:\n{out}")
        if verbose and asm is None and out.strip():
            print(out)
        if asm is not None:
            _check_no_packed_fp32(asm, src)
            _check_stream_stores(asm, src)
            _check_m0_loads(asm, src)
            _check_cached_stores(asm, src)
            os.remove(asm)
    tmp = LIB_PATH + ".tmp"
    link = [hipcc(), "--offload-arch=gfx950", "-shared", "-fPIC", "-o", tmp, *objs]
    res = subprocess.run(link, stdout=subprocess.PIPE, stderr=subprocess.STDOUT)
    if res.returncode != 0:
        raise RuntimeError("link failed:\n" + res.stdout.decode())
    os.replace(tmp, LIB_PATH)
    out = bind_proc.communicate()[0].decode()
    if bind_proc.returncode != 0:
        raise RuntimeError(f"hipcc failed on {BINDING_SRC}:\n{out}")
    tmp = BINDING_PATH + ".tmp"
    res = subprocess.run(_binding_link_cmd(bind_obj, tmp), stdout=subprocess.PIPE, stderr=subprocess.STDOUT)
    if res.returncode != 0:
        raise RuntimeError("link of the PyTorch binding failed:\n" + res.stdout.decode())
    os.replace(tmp, BINDING_PATH)
    return LIB_PATH


if __name__ == "__main__":
    # run as a script, this directory heads sys.path and its platform.py would shadow the standard
    # library's `platform` for every later import (torch's included)
    sys.path = [p for p in sys.path if os.path.abspath(p or ".") != HERE]
    print(build(verbose="-v" in sys.argv))
