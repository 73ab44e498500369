"""Builds libmi355_layer.so (gfx950 only) from the HIP sources in this directory, and mi355_host.so, the Python
extension module with the native host path, from host.cpp.

Usage: python -m scaling_amd.csrc.build      (or scaling_amd.csrc.build.build() from Python)
Each .hip file is one translation unit; objects go to ./build/, the libraries next to the sources.
"""

import os
import shutil
import subprocess
import sys
import sysconfig
from concurrent.futures import ThreadPoolExecutor

HERE = os.path.dirname(os.path.abspath(__file__))
LIB_NAME = "libmi355_layer.so"
LIB_PATH = os.path.join(HERE, LIB_NAME)
HOST_NAME = "mi355_host"
HOST_PATH = os.path.join(HERE, HOST_NAME + ".so")
SOURCES = ["abi.hip", "rmsnorm.hip", "swiglu.hip", "rotary.hip", "attn_host.hip", "attn_fwd.hip", "attn_bwd.hip",
           "attn_decode.hip", "attn_f32.hip", "cross_entropy.hip", "gemm.hip", "gemm_wide.hip", "rows.hip"]
F16_SOURCES = ["attn_fwd.hip", "attn_bwd.hip", "attn_decode.hip"]
# packed fp32 VALU instructions stay disabled for every device translation unit; the kernels never
# produce NaNs on purpose (masked scores are -inf and every inf - inf is guarded), so NaN-preserving
# canonicalisation of the MFMA results before max / min is switched off
FLAGS = ["--offload-arch=gfx950", "-O3", "-std=c++17", "-fPIC", "-Xclang", "-target-feature", "-Xclang",
         "-packed-fp32-ops", "-fno-honor-nans", "-Wno-unused-command-line-argument"]


def _hipcc() -> str:
    exe = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not os.path.exists(exe):
        raise RuntimeError("hipcc not found; libmi355_layer.so cannot be built")
    return exe


def _run(cmd):
    proc = subprocess.run(cmd, cwd=HERE, capture_output=True, text=True)
    if proc.returncode != 0:
        raise RuntimeError("command failed: %s\n%s\n%s" % (" ".join(cmd), proc.stdout, proc.stderr))
    return proc


def build(verbose: bool = False, jobs: int = 8) -> str:
    hipcc = _hipcc()
    obj_dir = os.path.join(HERE, "build")
    os.makedirs(obj_dir, exist_ok=True)

    def compile_one(job):
        src, suffix, defines = job
        obj = os.path.join(obj_dir, src.replace(".hip", suffix + ".o"))
        _run([hipcc] + FLAGS + defines + ["-c", src, "-o", obj])
        if verbose:
            print("compiled", src, " ".join(defines), flush=True)
        return obj

    def compile_host(_job):
        import torch
        root = os.path.dirname(torch.__file__)
        obj = os.path.join(obj_dir, "host.o")
        includes = [os.path.join(root, "include"), os.path.join(root, "include", "torch", "csrc", "api", "include"), "/opt/rocm/include",
                    sysconfig.get_paths()["include"]]
        _run(["g++", "-O2", "-std=c++17", "-fPIC", "-D__HIP_PLATFORM_AMD__=1", "-DUSE_ROCM=1", "-DTORCH_API_INCLUDE_EXTENSION_H",
              f"-DTORCH_EXTENSION_NAME={HOST_NAME}", f"-D_GLIBCXX_USE_CXX11_ABI={int(torch.compiled_with_cxx11_abi())}"]
             + [f"-I{d}" for d in includes] + ["-c", "host.cpp", "-o", obj])
        if verbose:
            print("compiled host.cpp", flush=True)
        return obj, os.path.join(root, "lib")

    # the attention kernels exist once per element type: bfloat16 (as is) and float16 (-DMI_ELEM_F16)
    jobs_list = [(s, "", []) for s in SOURCES] + [(s, "_f16", ["-DMI_ELEM_F16"]) for s in F16_SOURCES]
    jobs_list.sort(key=lambda j: 0 if j[0] in ("attn_fwd.hip", "attn_bwd.hip") else 1)   # the slow ones first
    with ThreadPoolExecutor(max_workers=jobs) as pool:
        host = pool.submit(compile_host, None)
        objs = list(pool.map(compile_one, jobs_list))
        host_obj, torch_lib = host.result()
    tmp = LIB_PATH + ".tmp"
    _run([hipcc, "--offload-arch=gfx950", "-shared", "-fPIC", "-o", tmp] + objs)
    os.replace(tmp, LIB_PATH)
    tmp = HOST_PATH + ".tmp"
    _run(["g++", "-shared", "-o", tmp, host_obj, f"-L{torch_lib}", "-lc10", "-lc10_hip", "-ltorch", "-ltorch_cpu", "-ltorch_hip",
          "-ltorch_python", f"-L{HERE}", f"-l:{LIB_NAME}", "-Wl,-rpath,$ORIGIN"])
    os.replace(tmp, HOST_PATH)
    if verbose:
        print("linked", LIB_PATH, HOST_PATH, flush=True)
    return LIB_PATH


if __name__ == "__main__":
    build(verbose=True)
    sys.exit(0)
