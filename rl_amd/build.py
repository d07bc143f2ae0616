"""Builds ``librl_amd_hip.so`` (the C-ABI HIP library) for gfx950 with hipcc and ``_host.so`` (the host side of the calls,
plain C++ against PyTorch) with g++.

``python -m rl_amd.build`` compiles every ``csrc/*.hip`` and ``csrc/host_path.cpp`` into ``rl_amd/lib/``.  hipcc
cross-compiles without a GPU.  Packed-FP32 instruction selection is switched off for all
device code.
"""

from __future__ import annotations

import glob
import os
import subprocess
import sys

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
LIB_DIR = os.path.join(HERE, "lib")
ROCM = os.environ.get("ROCM_PATH", "/opt/rocm")
LIB_PATH = os.path.join(LIB_DIR, "librl_amd_hip.so")
HOST_PATH = os.path.join(LIB_DIR, "_host.so")

HIPCC_FLAGS = [
    "-O3",
    "--offload-arch=gfx950",
    "-std=c++17",
    "-fPIC",
    "-ffp-contract=off",  # token arithmetic mirrors separate fp32 PyTorch ops: no fused multiply-add
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
]


def sources() -> list[str]:
    return sorted(glob.glob(os.path.join(CSRC, "*.hip")))


def host_command(obj: str) -> list[str]:
    """g++ command line that compiles ``host_path.cpp`` to ``obj``."""
    import sysconfig

    import torch

    inc = os.path.join(os.path.dirname(torch.__file__), "include")
    dirs = [inc, os.path.join(inc, "torch", "csrc", "api", "include"), os.path.join(ROCM, "include"), sysconfig.get_paths()["include"]]
    return [os.environ.get("CXX", "g++"), "-O2", "-std=c++17", "-fPIC", "-fvisibility=hidden", "-D__HIP_PLATFORM_AMD__=1", "-DUSE_ROCM=1",
            f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}", "-DTORCH_EXTENSION_NAME=_host",
            *(a for d in dirs for a in ("-isystem", d)), "-c", os.path.join(CSRC, "host_path.cpp"), "-o", obj]


def link_host_command(obj: str) -> list[str]:
    import torch

    lib = os.path.join(os.path.dirname(torch.__file__), "lib")
    return [os.environ.get("CXX", "g++"), "-shared", "-o", HOST_PATH, obj, f"-L{lib}", "-ltorch", "-ltorch_cpu", "-ltorch_python", "-lc10",
            "-lc10_hip", "-ltorch_hip", f"-L{LIB_DIR}", "-l:librl_amd_hip.so", f"-L{ROCM}/lib", "-lamdhip64", "-Wl,-rpath,$ORIGIN"]


def build(verbose: bool = True) -> str:
    """Compile every HIP source and link the shared library, then the host extension; returns the library's path."""
    hipcc = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
    os.makedirs(LIB_DIR, exist_ok=True)
    objs = []
    procs = []
    host_obj = os.path.join(LIB_DIR, "host_path.o")
    cmd = host_command(host_obj)
    if verbose:
        print(" ".join(cmd), flush=True)
    procs.append((os.path.join(CSRC, "host_path.cpp"), subprocess.Popen(cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)))
    for src in sources():
        obj = os.path.join(LIB_DIR, os.path.basename(src)[:-4] + ".o")
        objs.append(obj)
        cmd = [hipcc, *HIPCC_FLAGS, "-c", src, "-o", obj]
        if verbose:
            print(" ".join(cmd), flush=True)
        procs.append((src, subprocess.Popen(cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)))
    failed = False
    for src, proc in procs:
        out, _ = proc.communicate()
        noise = "packed-fp32-ops"
        text = "\n".join(l for l in out.splitlines() if noise not in l and l.strip())
        if proc.returncode != 0:
            failed = True
            print(f"compilation failed for {src}:\n{out}", file=sys.stderr)
        elif verbose and text:
            print(text)
    if failed:
        raise RuntimeError("compilation failed")
    cmd = [hipcc, "--offload-arch=gfx950", "-shared", "-fPIC", "-o", LIB_PATH, *objs]
    if verbose:
        print(" ".join(cmd), flush=True)
    subprocess.run(cmd, check=True)
    cmd = link_host_command(host_obj)
    if verbose:
        print(" ".join(cmd), flush=True)
    subprocess.run(cmd, check=True)
    for obj in objs + [host_obj]:
        os.remove(obj)
    return LIB_PATH


if __name__ == "__main__":
    print(build())
