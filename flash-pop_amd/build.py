"""Builds flash_pop_amd/libflashpop_hip.so for gfx950 with hipcc (cross-compiles without a GPU) and, linked to it,
flash_pop_amd/_native.so, the PyTorch ops (host code only)."""
import os
import subprocess
import sys
import sysconfig

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
OUT = os.path.join(HERE, "flash_pop_amd", "libflashpop_hip.so")
NATIVE_OUT = os.path.join(HERE, "flash_pop_amd", "_native.so")
SOURCES = ["launch_hip.hip", "flashpop_api.cpp"]
FLAGS = ["--offload-arch=gfx950", "-O3", "-std=c++17", "-fPIC", "-shared",
         "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops"]


def _run(cmd, verbose):
    if verbose:
        print(" ".join(cmd), flush=True)
    res = subprocess.run(cmd, capture_output=True, text=True)
    # hipcc's host pass warns that it does not know the packed-fp32 feature; drop only that noise
    noise = "is not a recognized feature for this target"
    err = "\n".join(l for l in res.stderr.splitlines() if noise not in l)
    if err.strip() and (verbose or res.returncode):
        print(err, file=sys.stderr)
    if res.returncode != 0:
        raise RuntimeError(f"{cmd[0]} failed with exit code {res.returncode}")


def native_command(out=NATIVE_OUT, library=OUT, device_dir=CSRC):
    """`library`: the C-ABI library to link; `device_dir`: where torch_device.h is found (the CPU tests have one of their own)."""
    import torch
    root = os.path.dirname(torch.__file__)
    rocm = os.environ.get("ROCM_PATH", "/opt/rocm")
    includes = [device_dir, f"{root}/include", f"{root}/include/torch/csrc/api/include", f"{rocm}/include", sysconfig.get_paths()["include"]]
    return ["g++", "-O2", "-std=c++17", "-fPIC", "-shared", "-D__HIP_PLATFORM_AMD__=1", "-DUSE_ROCM=1",
            f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}", *[a for i in includes for a in ("-isystem", i)],
            os.path.join(CSRC, "torch_ops.cpp"), "-o", out,
            "-L", os.path.dirname(library), "-l:" + os.path.basename(library), "-L", f"{root}/lib", "-ltorch_python", "-ltorch", "-ltorch_cpu",
            "-ltorch_hip", "-lc10", "-lc10_hip", "-Wl,-rpath,$ORIGIN", f"-Wl,-rpath,{root}/lib"]


def build(verbose: bool = True) -> str:
    _run(["hipcc", *FLAGS, *[os.path.join(CSRC, s) for s in SOURCES], "-o", OUT], verbose)
    _run(native_command(), verbose)
    return OUT


if __name__ == "__main__":
    print(build())
