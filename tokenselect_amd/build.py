"""Build ``libtokenselect_hip.so`` for gfx950 with hipcc, and the Python binding, in-tree.

``python -m tokenselect_amd.build`` compiles every ``csrc/*.hip`` translation
unit (in parallel) and links them into ``tokenselect_amd/libtokenselect_hip.so``;
``csrc/bind/ts_bind.cpp`` becomes ``tokenselect_amd/_ts_bind.so`` with the host
compiler and PyTorch's headers.  hipcc cross-compiles without a GPU, so this runs
on a CPU-only host.
"""

import glob
import os
import subprocess
import sys
import sysconfig
from concurrent.futures import ThreadPoolExecutor

PKG_DIR = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(PKG_DIR, "csrc")
BUILD_DIR = os.path.join(PKG_DIR, "csrc", "build")
LIB_PATH = os.path.join(PKG_DIR, "libtokenselect_hip.so")
BIND_SRC = os.path.join(CSRC, "bind", "ts_bind.cpp")
BIND_PATH = os.path.join(PKG_DIR, "_ts_bind.so")

ROCM = "/opt/rocm"
HIPCC = os.environ.get("HIPCC", f"{ROCM}/bin/hipcc")
ARCH = "gfx950"
# Packed-FP32 instruction selection is switched off for all device code.
CXXFLAGS = [
    f"--offload-arch={ARCH}", "-O3", "-fPIC", "-std=c++17", "-Wall", "-Wno-unused-function",
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
]
# Matrix instructions write to the vector registers, as the vector instructions that follow on
# their results want them; accumulators that are to live in the others are placed by hand.
# (An internal option of the compiler: one that does not know it refuses it, and the build stops
# there.  Without it the kernel is as correct and moves its logits between the two halves of the
# register file.)
# The selection's additions to one word of LDS come from one lane of a wavefront each, or are combined
# by the code itself: left alone they are one instruction, while the compiler otherwise turns each
# into a loop over the active lanes (0.15 us apiece where a workgroup runs it once; one request of
# 32K tokens 36.8 -> 35.9 us a layer).
SOURCE_FLAGS = {"ts_prefill.hip": ["-mllvm", "-amdgpu-mfma-vgpr-form=1"],
                "ts_prefill_chunks.hip": ["-mllvm", "-amdgpu-mfma-vgpr-form=1"],
                "ts_prefill_shared.hip": ["-mllvm", "-amdgpu-mfma-vgpr-form=1"],
                "ts_score.hip": ["-mllvm", "-amdgpu-atomic-optimizer-strategy=None"]}


def sources():
    return sorted(glob.glob(os.path.join(CSRC, "*.hip")))


def _compile(src: str, extra) -> str:
    obj = os.path.join(BUILD_DIR, os.path.basename(src)[:-4] + ".o")
    cmd = [HIPCC, *CXXFLAGS, *SOURCE_FLAGS.get(os.path.basename(src), ()), *extra, "-c", src, "-o", obj]
    res = subprocess.run(cmd, capture_output=True, text=True)
    if res.returncode != 0:
        raise RuntimeError(f"hipcc failed for {src}:\n{res.stdout}\n{res.stderr}")
    noise = "'-packed-fp32-ops' is not a recognized feature"
    warn = "\n".join(line for line in res.stderr.splitlines() if line and noise not in line)
    if warn.strip():
        sys.stderr.write(warn + "\n")
    return obj


def build_binding() -> str:
    """The binding has no device code: the host compiler, against the PyTorch that is installed."""
    import torch
    home = os.path.dirname(torch.__file__)
    tmp = BIND_PATH + ".tmp"
    cmd = [os.environ.get("CXX", "g++"), "-O2", "-fPIC", "-std=c++17", "-shared", "-Wall",
           "-D__HIP_PLATFORM_AMD__", "-DUSE_ROCM",
           f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}",
           "-isystem", os.path.join(home, "include"), "-isystem", os.path.join(ROCM, "include"),
           "-isystem", sysconfig.get_paths()["include"], BIND_SRC, "-o", tmp,
           "-L" + os.path.join(home, "lib"), "-lc10", "-lc10_hip", "-ltorch_cpu", "-ltorch_python"]
    res = subprocess.run(cmd, capture_output=True, text=True)
    if res.returncode != 0:
        raise RuntimeError(f"building the Python binding failed:\n{res.stdout}\n{res.stderr}")
    if res.stderr.strip():
        sys.stderr.write(res.stderr)
    os.replace(tmp, BIND_PATH)
    return BIND_PATH


def build(extra_flags=(), jobs: int = 8, verbose: bool = True) -> str:
    os.makedirs(BUILD_DIR, exist_ok=True)
    srcs = sources()
    if not srcs:
        raise RuntimeError(f"no .hip sources under {CSRC}")
    with ThreadPoolExecutor(max_workers=min(jobs, len(srcs) + 1)) as pool:
        binding = pool.submit(build_binding)
        objs = list(pool.map(lambda s: _compile(s, list(extra_flags)), srcs))
        binding.result()
    tmp = LIB_PATH + ".tmp"
    cmd = [HIPCC, f"--offload-arch={ARCH}", "-shared", "-fPIC", *objs, "-o", tmp]
    res = subprocess.run(cmd, capture_output=True, text=True)
    if res.returncode != 0:
        raise RuntimeError(f"link failed:\n{res.stdout}\n{res.stderr}")
    os.replace(tmp, LIB_PATH)
    if verbose:
        print(f"built {LIB_PATH} from {len(srcs)} translation units, and {BIND_PATH}")
    return LIB_PATH


if __name__ == "__main__":
    build(extra_flags=sys.argv[1:])
