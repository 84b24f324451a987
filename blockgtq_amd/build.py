"""Compile the gfx950 kernels into ``blockgtq_amd/_lib/libbgtq.so`` with hipcc.

hipcc cross-compiles without a GPU, so this runs anywhere the ROCm toolchain
is installed.  The library is kept in-tree next to the package.
"""
import os
import shutil
import subprocess
import sysconfig
from concurrent.futures import ThreadPoolExecutor

_HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(_HERE, "csrc")
LIB_DIR = os.path.join(_HERE, "_lib")
LIB_PATH = os.path.join(LIB_DIR, "libbgtq.so")
HOST_SRC = os.path.join(CSRC, "bgtq_host.cpp")
HOST_PATH = os.path.join(LIB_DIR, "_bgtq_host.so")       # CPython extension next to the library it calls

ARCH = "gfx950"
COMMON = ["--offload-arch=" + ARCH, "-O3", "-fPIC", "-std=c++17",
          "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
          "-fhip-fp32-correctly-rounded-divide-sqrt",
          # leading scalar arguments of a kernel are in registers when its waves start, instead of a trip to memory away
          "-mllvm", "-amdgpu-kernarg-preload-count=16"]
# source file -> extra flags.  The encoders promise a fixed floating-point
# evaluation order, so nothing in that file may be contracted into an fma
# behind the author's back.
SOURCES = {
    "bgtq_encode.hip": ["-ffp-contract=off", "-fno-strict-aliasing"],
    "bgtq_decode.hip": ["-fno-strict-aliasing"],
    # LDS tiles are written as 128-bit / 16-bit words and read back as 32-bit words
    "bgtq_decode_seg.hip": ["-fno-strict-aliasing"],
    "bgtq_dequant.hip": [],
    "bgtq_prefill.hip": ["-fno-strict-aliasing"],
    "bgtq_prompt.hip": ["-fno-strict-aliasing"],
}


def _hipcc():
    exe = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not os.path.exists(exe):
        raise RuntimeError("hipcc not found; the kernels need the ROCm toolchain")
    return exe


def _run(cmd, what, verbose):
    if verbose:
        print(" ".join(cmd), flush=True)
    res = subprocess.run(cmd, capture_output=True, text=True)
    if res.returncode != 0:
        raise RuntimeError(f"{what} failed:\n{res.stderr}")


def _host_command(out):
    """Compile line of the CPython extension: host code only, against the torch that will import it."""
    from torch.utils import cpp_extension
    includes = cpp_extension.include_paths("cuda") + [sysconfig.get_paths()["include"]]
    torch_lib = cpp_extension.library_paths("cuda")[0]
    return ([shutil.which("g++") or "g++", "-O2", "-std=c++17", "-fPIC", "-shared", "-D__HIP_PLATFORM_AMD__=1", "-DUSE_ROCM=1",
             "-fvisibility=hidden", "-w"] + ["-isystem" + p for p in includes] +
            [HOST_SRC, "-o", out, "-L" + LIB_DIR, "-L" + torch_lib, "-Wl,-rpath,$ORIGIN",
             "-l:libbgtq.so", "-ltorch_python", "-ltorch_cpu", "-ltorch", "-lc10", "-lc10_hip"])


def build(verbose=False):
    """Compile every HIP source, link the shared library and compile the CPython extension that
    calls it.  Returns the library's path."""
    hipcc = _hipcc()
    os.makedirs(LIB_DIR, exist_ok=True)
    objs = [os.path.join(LIB_DIR, src.replace(".hip", ".o")) for src in SOURCES]
    with ThreadPoolExecutor(len(SOURCES)) as pool:
        jobs = [pool.submit(_run, [hipcc] + COMMON + extra + ["-c", os.path.join(CSRC, src), "-o", obj], f"hipcc on {src}", verbose)
                for (src, extra), obj in zip(SOURCES.items(), objs)]
        for j in jobs:
            j.result()
    tmp = LIB_PATH + ".tmp"
    _run([hipcc, "--offload-arch=" + ARCH, "-shared", "-fPIC", "-Wl,-soname,libbgtq.so"] + objs + ["-o", tmp], "link", verbose)
    os.replace(tmp, LIB_PATH)
    tmp = HOST_PATH + ".tmp"
    _run(_host_command(tmp), "g++ on bgtq_host.cpp", verbose)
    os.replace(tmp, HOST_PATH)
    return LIB_PATH


if __name__ == "__main__":
    print(build(verbose=True))
