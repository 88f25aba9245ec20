"""Compile the HIP sources under csrc/ into libdflash_mi355.so (gfx950 only), and the native launch path
(csrc/host.cpp, host code against torch's headers) into _dflash_host.so beside it.

Usage: ``python build_ext.py`` (or ``build()`` from Python).  hipcc cross-compiles,
so no GPU is needed to build.
"""
from __future__ import annotations

import os
import subprocess
import sys

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)
CSRC = os.path.join(HERE, "csrc")
CSRC_INCLUDE = os.path.join(ROOT, "include")
LIB_PATH = os.path.join(HERE, "libdflash_mi355.so")
HOST_PATH = os.path.join(HERE, "_dflash_host.so")

SOURCES = ["api.hip", "qmm_m16.hip", "qmm_m16_stream.hip", "qmm_m16_chain.hip", "qmm_narrow.hip", "qmm_resident.hip", "qmm_resident_bf16.hip", "qmm_resident_fp16.hip", "qmm_resident_rows_bf16.hip", "qmm_resident_rows_fp16.hip", "qmm_resident_gather.hip", "qmm_rows.hip", "tape_replay.hip", "gdn_forward.hip", "gdn_prompt.hip", "gdn_glue.hip", "attn_glue.hip", "sdpa_q16.hip",
           "conv_state.hip"]

HIPCC_FLAGS = [
    "--offload-arch=gfx950",
    "-O3",
    "-std=c++17",
    "-fPIC",
    "-shared",
    "-fno-gpu-rdc",
    # scalar fp32 code only: keep the compiler from forming packed-fp32 VALU ops
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wall",
    "-Wno-unused-command-line-argument",
]


def _host_commands(obj: str) -> tuple:
    """Compile and link lines of the native launch path (``obj``: its object file)."""
    import sysconfig

    import torch
    from torch.utils import cpp_extension

    includes = [CSRC_INCLUDE, *cpp_extension.include_paths(), "/opt/rocm/include", sysconfig.get_paths()["include"]]
    compile_line = ["g++", "-O2", "-std=c++17", "-fPIC", "-Wall", "-D__HIP_PLATFORM_AMD__=1", "-DUSE_ROCM=1",
                    f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}", "-I", includes[0],
                    *(part for path in includes[1:] for part in ("-isystem", path)),
                    "-c", os.path.join(CSRC, "host.cpp"), "-o", obj]
    torch_lib = os.path.join(os.path.dirname(torch.__file__), "lib")
    link_line = ["g++", "-shared", obj, "-o", HOST_PATH + ".tmp", "-L", HERE, f"-l:{os.path.basename(LIB_PATH)}",
                 "-L", torch_lib, "-lc10", "-lc10_hip", "-ltorch_cpu", "-ltorch_python", "-Wl,-rpath,$ORIGIN"]
    return compile_line, link_line


def build(verbose: bool = False) -> str:
    """Every source to an object file of its own, side by side (the sources do not depend on each
    other's objects; one compiler run over all of them takes twice as long), then one link."""
    import tempfile
    from concurrent.futures import ThreadPoolExecutor

    hipcc = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
    flags = [f for f in HIPCC_FLAGS if f != "-shared"]
    jobs = max(1, min(len(SOURCES), int(os.environ.get("MAX_JOBS", "8"))))
    with tempfile.TemporaryDirectory() as tmp:
        def run(cmd: list) -> None:
            if verbose:
                print(" ".join(cmd), flush=True)
            subprocess.run(cmd, check=True)

        def compile_one(src: str) -> str:
            obj = os.path.join(tmp, src.replace(".hip", ".o"))
            run([hipcc, *flags, "-I", CSRC_INCLUDE, "-I", CSRC, "-c", os.path.join(CSRC, src), "-o", obj])
            return obj

        host_obj = os.path.join(tmp, "host.o")
        host_compile, host_link = _host_commands(host_obj)

        with ThreadPoolExecutor(max_workers=jobs) as pool:
            host = pool.submit(run, host_compile)
            objects = list(pool.map(compile_one, SOURCES))
            host.result()
        run([hipcc, "--offload-arch=gfx950", "-shared", "-fPIC", "-fno-gpu-rdc", *objects, "-o", LIB_PATH + ".tmp"])
        os.replace(LIB_PATH + ".tmp", LIB_PATH)
        run(host_link)
        os.replace(HOST_PATH + ".tmp", HOST_PATH)
    return LIB_PATH


if __name__ == "__main__":
    print(build(verbose="-v" in sys.argv))
