"""
Build recipe of libkvx.so (hipcc for gfx950 on the HIP sources under csrc/, linked into one shared library next to this
file) and of _host.so (the extension module of csrc/host.cpp, host code only, against the installed PyTorch).
Cross-compiles without a GPU. Run as `python -m keys_values_amd.build`.
"""
import os
import subprocess
import sys
import sysconfig
from concurrent.futures import ThreadPoolExecutor
from importlib.util import find_spec

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
OBJ = os.path.join(HERE, "build")
LIB = os.path.join(HERE, "libkvx.so")
HOST = os.path.join(HERE, "_host.so")
SOURCES = ["sdpa_decode_128.hip", "sdpa_decode_64.hip", "sdpa_decode_256.hip", "score_sum.hip", "sdpa_prefill.hip", "sdpa_rows.hip", "quantize.hip", "h2o.hip", "kvx_api.hip",
           "sdpa_decode.hip", "norm_rope.hip"]  # the longest first

HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
FLAGS = [
    "--offload-arch=gfx950",
    "-O3",
    "-std=c++17",
    "-fPIC",
    "-fno-fast-math",          # the quantiser relies on IEEE division and rounding
    "-ffp-contract=off",       # no implicit fused multiply-add; kernels call fmaf where they want one
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wall",
    "-Wno-unused-function",
    "-Wno-inline-asm",         # the DMA helpers name m0 as clobbered, which clang reports once per instantiation
]


def _compile(src: str) -> str:
    os.makedirs(OBJ, exist_ok=True)
    obj = os.path.join(OBJ, src.replace(".hip", ".o"))
    cmd = [HIPCC] + FLAGS + ["-c", os.path.join(CSRC, src), "-o", obj]
    res = subprocess.run(cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
    out = "\n".join(l for l in res.stdout.splitlines() if "packed-fp32-ops" not in l)
    if res.returncode != 0:
        raise RuntimeError(f"hipcc failed on {src}:\n{out}")
    if out.strip():
        print(out, file=sys.stderr)
    return obj


def _build_host():
    torch_dir = os.path.dirname(find_spec("torch").origin)
    rocm = os.path.dirname(os.path.dirname(HIPCC))
    cmd = [os.environ.get("CXX", "g++"), "-O2", "-std=c++17", "-fPIC", "-shared", "-Wall", "-D__HIP_PLATFORM_AMD__=1", "-DUSE_ROCM=1",
           "-I" + sysconfig.get_paths()["include"], "-isystem", os.path.join(rocm, "include"), "-isystem", os.path.join(torch_dir, "include"),
           "-isystem", os.path.join(torch_dir, "include", "torch", "csrc", "api", "include"), os.path.join(CSRC, "host.cpp"), "-o", HOST,
           "-L" + os.path.join(torch_dir, "lib"), "-ltorch_python", "-ltorch_cpu", "-ltorch_hip", "-lc10_hip", "-lc10", "-ldl"]
    res = subprocess.run(cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
    if res.returncode != 0:
        raise RuntimeError(f"g++ failed on host.cpp:\n{res.stdout}")


def build(verbose: bool = True) -> str:
    with ThreadPoolExecutor(max_workers=min(8, os.cpu_count() or 1)) as ex:
        host = ex.submit(_build_host)
        objs = list(ex.map(_compile, SOURCES))
        host.result()
    cmd = [HIPCC, "--offload-arch=gfx950", "-shared", "-fPIC", "-o", LIB] + objs
    res = subprocess.run(cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
    if res.returncode != 0:
        raise RuntimeError(f"link failed:\n{res.stdout}")
    if verbose:
        print(f"built {LIB}")
    return LIB


if __name__ == "__main__":
    build()
