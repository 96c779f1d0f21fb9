"""Compile the native parts next to their sources:

* libpbs_hip.so, the C-ABI HIP library, for gfx950;
* libpbs_hip_check.so: the same library with the conservative progress protocol of the two barrier-free bf16
  kernels (-DPBS_DDS16_PUBLISH_AFTER_WAIT -DPBS_DDSC_PUBLISH_AFTER_WAIT).  Only tests/test_gpu_wide_protocol.py loads it,
  to compare the two bit for bit;
* _pbs_torch.so, the extension module between torch and libpbs_hip.so (host code only).
"""
import os
import subprocess
import sys
import sysconfig
from concurrent.futures import ThreadPoolExecutor

HERE = os.path.dirname(os.path.abspath(__file__))
LIB = os.path.join(HERE, "libpbs_hip.so")
CHECK_LIB = os.path.join(HERE, "libpbs_hip_check.so")
TORCH_EXT = os.path.join(HERE, "_pbs_torch.so")


def build(verbose=True):
    with ThreadPoolExecutor(3) as pool:
        jobs = [pool.submit(_run, cmd, verbose) for cmd in (
            _hip_command(LIB, []),
            _hip_command(CHECK_LIB, ["-DPBS_DDS16_PUBLISH_AFTER_WAIT", "-DPBS_DDSC_PUBLISH_AFTER_WAIT"]),
            _torch_command(compile_only=True),
        )]
        for j in jobs:
            j.result()
    _link_torch(verbose)
    return LIB


def build_torch(verbose=True):
    """_pbs_torch.so alone, next to a libpbs_hip.so that is there (the Makefile's way)."""
    _run(_torch_command(compile_only=True), verbose)
    _link_torch(verbose)


def _link_torch(verbose):
    _run(_torch_command(compile_only=False), verbose)   # links against libpbs_hip.so
    os.remove(TORCH_EXT + ".o")


def _hip_command(lib, defines):
    return [
        os.environ.get("HIPCC", "hipcc"),
        "-O3",
        "-std=c++17",
        "--offload-arch=gfx950",
        "-fPIC",
        "-shared",
        "-Xclang",
        "-target-feature",
        "-Xclang",
        "-packed-fp32-ops",
        *defines,
        "-o",
        lib,
        os.path.join(HERE, "pbs_hip.hip"),
    ]


def _torch_command(compile_only):
    import torch
    from torch.utils.cpp_extension import include_paths, library_paths

    cxx = os.environ.get("CXX", "g++")
    if not compile_only:
        return [cxx, "-shared", TORCH_EXT + ".o", "-o", TORCH_EXT, "-L" + HERE, "-l:libpbs_hip.so",
                *("-L" + p for p in library_paths(device_type="cuda")), "-ltorch", "-ltorch_cpu", "-ltorch_hip", "-lc10", "-lc10_hip",
                "-ltorch_python", "-Wl,-rpath,$ORIGIN"]
    paths = include_paths(device_type="cuda") + [sysconfig.get_paths()["include"]]
    return [cxx, "-O2", "-std=c++17", "-fPIC", "-c", "-D__HIP_PLATFORM_AMD__=1", "-DUSE_ROCM",
            "-D_GLIBCXX_USE_CXX11_ABI=%d" % torch._C._GLIBCXX_USE_CXX11_ABI, *(a for p in paths for a in ("-isystem", p)),
            os.path.join(HERE, "pbs_torch.cpp"), "-o", TORCH_EXT + ".o"]


def _run(cmd, verbose):
    if verbose:
        print(" ".join(cmd), flush=True)
    res = subprocess.run(cmd, cwd=HERE, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
    # the host pass of hipcc prints one harmless "not a recognized feature" line per compile step
    out = "\n".join(l for l in res.stdout.splitlines() if "packed-fp32-ops" not in l)
    if out.strip() and verbose:
        print(out)
    if res.returncode != 0:
        raise RuntimeError("%s failed:\n%s" % (cmd[0], res.stdout))


if __name__ == "__main__":
    build_torch() if "--torch-only" in sys.argv else build()
    sys.exit(0)
