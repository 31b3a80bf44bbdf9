"""Build libbvllm_amd.so (the C-ABI HIP library) and the wrappers' native host side in-tree.

Usage: python baby-vllm_amd/build_lib.py [--jobs N]

Compiles every csrc/*.hip with hipcc for gfx950 only and links one shared
library next to the Python package (babyvllm/libbvllm_amd.so), and compiles
csrc/fast_calls.cpp (host code only) into the extension module
babyvllm/_fast_calls. The built files are what the wrappers load; they are not
tracked by git but travel with the tree.
"""

from __future__ import annotations

import argparse
import concurrent.futures as cf
import os
import subprocess
import sys
import sysconfig
from pathlib import Path

PKG_ROOT = Path(__file__).resolve().parent
CSRC = PKG_ROOT / "csrc"
INCLUDE = PKG_ROOT.parent / "include"
OUT = PKG_ROOT / "babyvllm" / "libbvllm_amd.so"
OBJ_DIR = PKG_ROOT / "_build"
FAST_OUT = PKG_ROOT / "babyvllm" / ("_fast_calls" + sysconfig.get_config_var("EXT_SUFFIX"))

HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
ARCH = "gfx950"
FLAGS = [
    f"--offload-arch={ARCH}",
    "-O3",
    "-std=c++17",
    "-fPIC",
    "-fvisibility=hidden",
    "-Wall",
    "-Wno-unused-function",
    "-I", str(INCLUDE),
    # Packed-FP32 VALU forms are kept out of the generated code.
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
]


# Per-file additions: paged_decode_pair.hip keeps its MFMA accumulators in
# VGPRs (see the file's header for the measurements).
FILE_FLAGS = {
    "paged_decode_pair.hip": ["-mllvm", "-amdgpu-mfma-vgpr-form"],
}


def _compile(src: Path) -> Path:
    obj = OBJ_DIR / (src.stem + ".o")
    cmd = [HIPCC, *FLAGS, *FILE_FLAGS.get(src.name, []), "-c", str(src), "-o", str(obj)]
    res = subprocess.run(cmd, capture_output=True, text=True)
    noise = "is not a recognized feature for this target"
    err = "\n".join(l for l in res.stderr.splitlines() if noise not in l)
    if res.returncode != 0:
        raise RuntimeError(f"hipcc failed for {src.name}:\n{err}")
    if err.strip():
        print(err, file=sys.stderr)
    return obj


def build_fast_calls() -> Path:
    """The extension module of the wrappers' common calls (host code, built against torch)."""
    import torch
    from torch.utils import cpp_extension

    tmp = FAST_OUT.with_suffix(".so.tmp")
    cmd = [os.environ.get("CXX", "g++"), "-O2", "-std=c++17", "-fPIC", "-shared", "-fvisibility=hidden", "-Wall",
           f"-D_GLIBCXX_USE_CXX11_ABI={int(torch.compiled_with_cxx11_abi())}",
           "-isystem", sysconfig.get_paths()["include"],
           *(a for p in cpp_extension.include_paths() for a in ("-isystem", p)),
           str(CSRC / "fast_calls.cpp"), "-o", str(tmp),
           "-L", cpp_extension.TORCH_LIB_PATH, "-ltorch_python", "-ltorch_cpu", "-lc10"]
    res = subprocess.run(cmd, capture_output=True, text=True)
    if res.returncode != 0:
        raise RuntimeError(f"building fast_calls.cpp failed:\n{res.stderr}")
    if res.stderr.strip():
        print(res.stderr, file=sys.stderr)
    os.replace(tmp, FAST_OUT)
    return FAST_OUT


def build(jobs: int = 4) -> Path:
    OBJ_DIR.mkdir(exist_ok=True)
    sources = sorted(CSRC.glob("*.hip"))
    with cf.ThreadPoolExecutor(max_workers=max(1, jobs) + 1) as ex:
        fast = ex.submit(build_fast_calls)
        objs = list(ex.map(_compile, sources))
        fast.result()
    tmp = OUT.with_suffix(".so.tmp")
    cmd = [HIPCC, f"--offload-arch={ARCH}", "-shared", "-fPIC", "-o", str(tmp), *map(str, objs)]
    res = subprocess.run(cmd, capture_output=True, text=True)
    if res.returncode != 0:
        raise RuntimeError(f"link failed:\n{res.stderr}")
    os.replace(tmp, OUT)
    return OUT


def main() -> None:
    ap = argparse.ArgumentParser()
    ap.add_argument("--jobs", type=int, default=4)
    args = ap.parse_args()
    print(build(args.jobs))


if __name__ == "__main__":
    main()
