"""Build librglru_hip.so (hand-written gfx950 kernels + the C ABI) in-tree with hipcc, and _native.so (the PyTorch
operators over it, host code only) with the host compiler.

    python -m griffin_amd.build            # compile griffin_amd/librglru_hip.so and griffin_amd/_native.so

hipcc cross-compiles without a GPU present, so this runs on a CPU-only machine.
"""

from __future__ import annotations

import os
import shutil
import subprocess
import sys
import sysconfig
import tempfile
from concurrent.futures import ThreadPoolExecutor

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
LIB_NAME = "librglru_hip.so"
LIB_PATH = os.path.join(HERE, LIB_NAME)
SOURCES = ["rglru_scan.hip", "rglru_fused.hip", "rglru_fwd_rows.hip", "rglru_fused_bwd.hip", "rglru_decode.hip", "rglru_decode_linear.hip",
           "rglru_gate_gemm.hip", "rglru_linear.hip", "rglru_linear16.hip", "rglru_block_ops.hip", "rglru_tokens.hip"]
NATIVE_PATH = os.path.join(HERE, "_native.so")
NATIVE_SOURCE = "torch_ops.cpp"
ARCH = "gfx950"


def hipcc_path() -> str:
    found = shutil.which("hipcc")
    if found:
        return found
    candidate = os.path.join(os.environ.get("ROCM_PATH", "/opt/rocm"), "bin", "hipcc")
    if os.path.exists(candidate):
        return candidate
    raise RuntimeError("hipcc not found: the RG-LRU HIP library cannot be built")


def _native_commands(obj: str, out: str) -> tuple[list[str], list[str]]:
    """Compile and link lines of the operator module.  It finds librglru_hip.so next to itself ($ORIGIN)."""
    import torch                                             # its headers and libraries, found through the package

    root = torch.__path__[0]
    rocm = os.environ.get("ROCM_PATH", "/opt/rocm")
    compiler = shutil.which("g++") or os.path.join(rocm, "llvm", "bin", "clang++")
    compile_line = [
        compiler, "-c", "-O2", "-std=c++17", "-fPIC", "-w", "-D__HIP_PLATFORM_AMD__=1", "-DUSE_ROCM=1",
        "-DTORCH_API_INCLUDE_EXTENSION_H", f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}",
        "-I", os.path.join(root, "include"), "-I", os.path.join(root, "include", "torch", "csrc", "api", "include"),
        "-I", os.path.join(rocm, "include"), "-I", sysconfig.get_path("include"), os.path.join(CSRC, NATIVE_SOURCE), "-o", obj,
    ]
    link_line = [
        compiler, "-shared", obj, "-o", out, "-L", HERE, f"-l:{LIB_NAME}", "-L", os.path.join(root, "lib"), "-ltorch_python",
        "-ltorch", "-ltorch_cpu", "-ltorch_hip", "-lc10", "-lc10_hip", "-Wl,-rpath,$ORIGIN",
    ]
    return compile_line, link_line


def build(verbose: bool = False) -> str:
    """Compile every kernel for gfx950, link the shared library and the operator module over it; returns the
    library's path."""
    flags = [
        "-O3", "-std=c++17", "-fPIC", f"--offload-arch={ARCH}",
        "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
        "-Wno-unused-command-line-argument", "-ffp-contract=off", "-fno-strict-aliasing",
        "-I", os.path.join(os.path.dirname(HERE), "include"),
    ]
    noise = "is not a recognized feature for this target"
    logs: list[str] = []

    def run(cmd: list[str]) -> None:
        if verbose:
            print(" ".join(cmd))
        proc = subprocess.run(cmd, capture_output=True, text=True)
        log = "\n".join(line for line in (proc.stdout + proc.stderr).splitlines() if noise not in line)
        if proc.returncode != 0:
            raise RuntimeError(f"{os.path.basename(cmd[0])} failed:\n" + log)
        if log.strip():
            logs.append(log)

    # one object per source, compiled side by side, then one link
    tmp = LIB_PATH + ".tmp"
    with tempfile.TemporaryDirectory(prefix="rglru_build_") as objdir:
        objects = [os.path.join(objdir, os.path.splitext(s)[0] + ".o") for s in SOURCES]
        native_obj, native_tmp = os.path.join(objdir, "torch_ops.o"), NATIVE_PATH + ".tmp"
        native_compile, native_link = _native_commands(native_obj, native_tmp)
        jobs = [native_compile] + [[hipcc_path(), *flags, "-c", os.path.join(CSRC, s), "-o", o] for s, o in zip(SOURCES, objects)]
        with ThreadPoolExecutor(max_workers=min(len(jobs), os.cpu_count() or 1)) as pool:
            list(pool.map(run, jobs))
        run([hipcc_path(), "-shared", "-fPIC", f"--offload-arch={ARCH}", *objects, "-o", tmp])
        # A kernel template whose body the host pass cannot instantiate (seen with a target builtin called directly in a
        # __global__ template) loses its launch stub without any diagnostic; the library then links but does not load.
        missing = [line.split()[-1] for line in
                   subprocess.run(["nm", "-D", "--undefined-only", tmp], capture_output=True, text=True).stdout.splitlines()
                   if "__device_stub__" in line]
        if missing:
            os.remove(tmp)
            raise RuntimeError("hipcc produced a library with undefined kernel stubs (would not load): " + ", ".join(missing[:4]))
        os.replace(tmp, LIB_PATH)
        run(native_link)
        os.replace(native_tmp, NATIVE_PATH)
    if verbose and logs:
        print("\n".join(logs))
    return LIB_PATH


if __name__ == "__main__":
    print(build(verbose="-v" in sys.argv))
