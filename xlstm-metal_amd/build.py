"""Builds libxlstm_hip.so for gfx950 from csrc/*.hip and libxlstm_torch.so, the torch operators around it,
from csrc/torch_ops.cpp (in-tree, no JIT cache).

    python xlstm-metal_amd/build.py            # build (always recompiles)
    python xlstm-metal_amd/build.py --jobs 8

Objects go to xlstm-metal_amd/_build/, the libraries to
xlstm-metal_amd/xlstm_hip/lib/ (git-ignored; they travel to the GPU box with
the tree).
"""

from __future__ import annotations

import argparse
import concurrent.futures as cf
import os
import shutil
import subprocess
import sys

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
BUILD = os.path.join(HERE, "_build")
LIBDIR = os.path.join(HERE, "xlstm_hip", "lib")
LIB = os.path.join(LIBDIR, "libxlstm_hip.so")
OPS_LIB = os.path.join(LIBDIR, "libxlstm_torch.so")
OPS_SRC = os.path.join(CSRC, "torch_ops.cpp")
INCLUDE = os.path.join(os.path.dirname(HERE), "include")
ARCH = "gfx950"

CXXFLAGS = [
    f"--offload-arch={ARCH}", "-O3", "-std=c++17", "-fPIC", f"-I{INCLUDE}", f"-I{CSRC}",
    # keep the compiler from forming packed-fp32 VALU ops
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wno-unused-command-line-argument",
]


# Per-source compiler options.  chunkwise_fused.hip: LLVM's iterative ILP scheduler orders the
# fused kernel's MFMA / LDS / VALU streams better than the default (cfg2 prefill 0.553 -> 0.544 ms
# over six alternating runs on one box).  (It crashes the compiler on chunkwise_bwd.hip.)
EXTRA_FLAGS = {
    "chunkwise_fused.hip": ["-mllvm", "-amdgpu-sched-strategy=iterative-ilp"],
    "chunkwise_pipe.hip": ["-mllvm", "-amdgpu-sched-strategy=iterative-ilp"],
}


def hipcc() -> str:
    for cand in (os.environ.get("HIPCC"), "/opt/rocm/bin/hipcc", shutil.which("hipcc")):
        if cand and os.path.exists(cand):
            return cand
    raise RuntimeError("hipcc not found (looked at $HIPCC, /opt/rocm/bin/hipcc, PATH)")


def _compile(src: str) -> str:
    obj = os.path.join(BUILD, os.path.splitext(os.path.basename(src))[0] + ".o")
    cmd = [hipcc(), *CXXFLAGS, *EXTRA_FLAGS.get(os.path.basename(src), []), "-c", src, "-o", obj]
    res = subprocess.run(cmd, capture_output=True, text=True)
    noise = "is not a recognized feature for this target"
    err = "\n".join(l for l in (res.stderr or "").splitlines() if noise not in l)
    if res.returncode != 0:
        raise RuntimeError(f"compile failed: {' '.join(cmd)}\n{err}")
    if err.strip():
        sys.stderr.write(err + "\n")
    return obj


def _compile_ops() -> str:
    """Host code only: g++ against torch's headers (torch's own libraries are in the process already)."""
    import torch
    from torch.utils.cpp_extension import include_paths
    obj = os.path.join(BUILD, "torch_ops.o")
    cmd = ["g++", "-O2", "-std=c++17", "-fPIC", "-D__HIP_PLATFORM_AMD__=1", "-DUSE_ROCM=1",
           f"-D_GLIBCXX_USE_CXX11_ABI={int(torch.compiled_with_cxx11_abi())}", f"-I{INCLUDE}",
           *[f"-isystem{d}" for d in include_paths("cuda")], "-isystem/opt/rocm/include", "-c", OPS_SRC, "-o", obj]
    res = subprocess.run(cmd, capture_output=True, text=True)
    if res.returncode != 0:
        raise RuntimeError(f"compile failed: {' '.join(cmd)}\n{res.stderr}")
    return obj


def _link(cmd: list[str]) -> None:
    res = subprocess.run(cmd, capture_output=True, text=True)
    if res.returncode != 0:
        raise RuntimeError(f"link failed: {' '.join(cmd)}\n{res.stderr}")


def _link_ops(obj: str, libdir: str, out: str) -> None:
    import torch
    tlib = os.path.join(os.path.dirname(torch.__file__), "lib")
    _link(["g++", "-shared", "-fPIC", "-o", out, obj, f"-L{libdir}", "-lxlstm_hip", "-Wl,-rpath,$ORIGIN", f"-L{tlib}",
           "-ltorch", "-ltorch_cpu", "-lc10", "-lc10_hip", "-Wl,--no-as-needed"])


def build(jobs: int | None = None, verbose: bool = True) -> str:
    os.makedirs(BUILD, exist_ok=True)
    os.makedirs(LIBDIR, exist_ok=True)
    srcs = sorted(os.path.join(CSRC, f) for f in os.listdir(CSRC) if f.endswith(".hip"))
    jobs = jobs or min(8, len(srcs))
    with cf.ThreadPoolExecutor(max_workers=jobs) as ex:
        ops = ex.submit(_compile_ops)
        objs = list(ex.map(_compile, srcs))
        ops_obj = ops.result()
    # both linked before either is replaced: a failed link leaves the pair that was there
    new = os.path.join(BUILD, "lib")
    os.makedirs(new, exist_ok=True)
    lib, ops_lib = os.path.join(new, os.path.basename(LIB)), os.path.join(new, os.path.basename(OPS_LIB))
    _link([hipcc(), f"--offload-arch={ARCH}", "-shared", "-fPIC", "-o", lib, *objs])
    _link_ops(ops_obj, new, ops_lib)
    os.replace(lib, LIB)
    os.replace(ops_lib, OPS_LIB)
    if verbose:
        print(f"built {LIB} from {len(srcs)} sources and {OPS_LIB}")
    return LIB


def main() -> None:
    ap = argparse.ArgumentParser()
    ap.add_argument("--jobs", type=int, default=None)
    args = ap.parse_args()
    build(args.jobs)


if __name__ == "__main__":
    main()
