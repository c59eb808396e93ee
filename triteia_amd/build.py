"""Build recipe for libtriteia_hip.so (gfx950) and the torch binding of its ops -- run as `python -m triteia_amd.build`.

hipcc cross-compiles without a GPU, so this works in a CPU-only container.  Both are built in-tree:
triteia_amd/lib/libtriteia_hip.so (kernels and C ABI) and triteia_amd/lib/triteia_torch.so (host code only).
"""
import os
import subprocess
import sys
import sysconfig

HERE = os.path.dirname(os.path.abspath(__file__))
SRC = os.path.join(HERE, "csrc", "triteia_hip.hip")
LIB_DIR = os.path.join(HERE, "lib")
LIB = os.path.join(LIB_DIR, "libtriteia_hip.so")
TORCH_SRC = os.path.join(HERE, "csrc", "torch_ops.cpp")
TORCH_LIB = os.path.join(LIB_DIR, "triteia_torch.so")

HIPCC_FLAGS = [
    "--offload-arch=gfx950",
    "-O3",
    "-std=c++17",
    "-fPIC",
    "-shared",
    "-fvisibility=hidden",
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wno-unused-command-line-argument",
]


# The wide kernels wait for their direct-to-LDS loads with hand-counted `s_waitcnt vmcnt(N)`: N counts
# the loads the compiler emits behind them in program order.  The counts were checked against the assembly
# output of this compiler; another one may order or split the loads differently, so the build refuses it
# unless TRITEIA_HIP_ANY_COMPILER=1 says that the counts have been checked again (`-S`, then the GPU parity tests).
VERIFIED_COMPILER = "roc-7.2.0"


def check_compiler(hipcc: str) -> str:
    out = subprocess.run([hipcc, "--version"], capture_output=True, text=True).stdout
    if VERIFIED_COMPILER not in out and os.environ.get("TRITEIA_HIP_ANY_COMPILER") != "1":
        raise RuntimeError(
            f"{hipcc} is not the compiler the hand-counted waits were verified with ({VERIFIED_COMPILER}):\n{out}"
            "set TRITEIA_HIP_ANY_COMPILER=1 after checking them again")
    return out


def build(verbose: bool = True, extra_flags=()) -> str:
    os.makedirs(LIB_DIR, exist_ok=True)
    hipcc = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
    check_compiler(hipcc)
    cmd = [hipcc, *HIPCC_FLAGS, *extra_flags, "-o", LIB, SRC]
    if verbose:
        print("[triteia_amd.build]", " ".join(cmd), flush=True)
    res = subprocess.run(cmd, capture_output=True, text=True)
    # the host pass does not know the gfx950-only feature flag and says so; drop that line
    noise = "is not a recognized feature for this target"
    err = "\n".join(l for l in res.stderr.splitlines() if noise not in l)
    if res.returncode != 0:
        raise RuntimeError(f"hipcc failed ({res.returncode}):\n{err}")
    if verbose and err.strip():
        print(err, file=sys.stderr)
    build_torch_binding(verbose=verbose)
    return LIB


def build_torch_binding(verbose: bool = True) -> str:
    """The ops' native call path (host code, no device code): g++ against the installed torch and the library above."""
    import torch
    root = os.path.dirname(torch.__file__)
    rocm = os.environ.get("ROCM_PATH", "/opt/rocm")
    cmd = ["g++", "-O2", "-std=c++17", "-fPIC", "-shared", "-fvisibility=hidden", "-D__HIP_PLATFORM_AMD__=1", "-DUSE_ROCM=1",
           f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}", f"-I{root}/include",
           f"-I{root}/include/torch/csrc/api/include", f"-I{rocm}/include", f"-I{sysconfig.get_paths()['include']}", TORCH_SRC, "-o", TORCH_LIB,
           f"-L{root}/lib", "-ltorch_python", "-ltorch", "-ltorch_cpu", "-ltorch_hip", "-lc10", "-lc10_hip", f"-L{LIB_DIR}", "-ltriteia_hip",
           "-Wl,-rpath,$ORIGIN"]
    if verbose:
        print("[triteia_amd.build]", " ".join(cmd), flush=True)
    res = subprocess.run(cmd, capture_output=True, text=True)
    if res.returncode != 0:
        raise RuntimeError(f"g++ failed ({res.returncode}):\n{res.stderr}")
    return TORCH_LIB


def ensure_built(verbose: bool = True) -> str:
    """The built library's path; compiles it (and the torch binding) first if (and only if) it is not in the tree.  For
    tests, smoke runs and benchmarks, which load what is built; `build()` itself compiles every time."""
    if not os.path.exists(LIB):
        build(verbose=verbose)
    elif not os.path.exists(TORCH_LIB):
        build_torch_binding(verbose=verbose)
    return LIB


if __name__ == "__main__":
    print(build(extra_flags=sys.argv[1:]))
