"""Build libmorph_optim.so for gfx950 and the host extension in-tree (python -m morph_amd.build).

Flags that matter for results:
  -ffp-contract=off       no implicit multiply-add fusion: the kernels round
                          exactly where torch's CPU kernels round, and fuse
                          only where __fmaf_rn says so;
  -packed-fp32-ops off    no packed FP32 instructions in device code.
  -fhip-fp32-correctly-rounded-divide-sqrt
                          fp32 `/` and sqrt lower to IEEE correctly
                          rounded sequences (hipcc's default, made explicit).
"""
import os
import subprocess
import sys
import sysconfig
from concurrent.futures import ThreadPoolExecutor
from pathlib import Path

PKG = Path(__file__).resolve().parent
ROOT = PKG.parent
SOURCES = ["abi.hip", "adamw.hip", "nonfinite.hip", "step.hip", "grads.hip", "convert.hip", "fp8.hip", "gemm.hip", "muon.hip", "muon_small.hip", "hostcopy.hip"]
OUTPUT = PKG / "lib" / "libmorph_optim.so"
HOSTPATH = PKG / "lib" / "_hostpath.so"  # Python extension over torch's C++ tensors (hostpath.cpp)
ARCH = os.environ.get("MORPH_OFFLOAD_ARCH", "gfx950")

FLAGS = [
    f"--offload-arch={ARCH}", "-O3", "-std=c++17", "-fPIC", "-shared",
    "-ffp-contract=off", "-fhip-fp32-correctly-rounded-divide-sqrt",
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    f"-I{ROOT / 'include'}",
    "-Werror=align-mismatch",  # a pointer passed on with a larger alignment than its type has
]


def hipcc():
    rocm = os.environ.get("ROCM_PATH", "/opt/rocm")
    return str(Path(rocm) / "bin" / "hipcc")


def build_hostpath(output=HOSTPATH):
    import torch
    from torch.utils import cpp_extension
    output = Path(output)
    output.parent.mkdir(parents=True, exist_ok=True)
    tmp = output.with_name(output.name + ".tmp")
    cmd = ["g++", "-O2", "-std=c++17", "-fPIC", "-shared", "-fvisibility=hidden",
           f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}",
           *[f"-isystem{p}" for p in cpp_extension.include_paths()],
           f"-isystem{sysconfig.get_paths()['include']}", "-o", str(tmp),
           str(PKG / "csrc" / "hostpath.cpp"), f"-L{Path(torch.__file__).parent / 'lib'}",
           "-lc10", "-ltorch_cpu", "-ltorch_python"]
    proc = subprocess.run(cmd, capture_output=True, text=True)
    if proc.returncode != 0:
        sys.stderr.write(proc.stdout + proc.stderr)
        raise RuntimeError(f"g++ failed ({proc.returncode}): {' '.join(cmd)}")
    os.replace(tmp, output)
    return output


def build_all():
    """The library and the host extension, compiled side by side."""
    with ThreadPoolExecutor(2) as pool:
        host = pool.submit(build_hostpath)
        library = build(quiet=False)
        return library, host.result()


def build(output=OUTPUT, extra_flags=(), quiet=True):
    output = Path(output)
    output.parent.mkdir(parents=True, exist_ok=True)
    tmp = output.with_name(output.name + ".tmp")
    cmd = [hipcc(), *FLAGS, *extra_flags, "-o", str(tmp),
           *[str(PKG / "csrc" / s) for s in SOURCES]]
    proc = subprocess.run(cmd, capture_output=True, text=True)
    if proc.returncode != 0:
        sys.stderr.write(proc.stdout + proc.stderr)
        raise RuntimeError(f"hipcc failed ({proc.returncode}): {' '.join(cmd)}")
    if not quiet:
        # The host pass warns that it does not know the packed-fp32 feature; drop that noise.
        noise = "is not a recognized feature for this target"
        sys.stderr.write("".join(l + "\n" for l in proc.stderr.splitlines() if noise not in l))
    os.replace(tmp, output)
    return output


if __name__ == "__main__":
    print(*build_all())
