"""Build libtaomate_h3_amd.so (gfx950) from csrc/ with hipcc, and the native
tensor wrappers (_h3q_torch.so) that call it with g++, in-tree.

    python taomate-h3_amd/build.py

The library exports only the C ABI of include/taomate_h3_amd.h.  Every HIP
source is compiled for gfx950 with packed-FP32 instruction selection off.
"""

from __future__ import annotations

import os
import shutil
import subprocess
import sys
import sysconfig
from concurrent.futures import ThreadPoolExecutor
from pathlib import Path

PKG = Path(__file__).resolve().parent
CSRC = PKG / "csrc"
LIB = PKG / "libtaomate_h3_amd.so"
# Measurement kernels of bench.py's `ceilings` object, kept out of the product library.
CEILINGS_SRC = "ceilings.hip"
CEILINGS_LIB = PKG / "libh3q_ceilings.so"
SOURCES = ["act_quant.hip", "head_quant.hip", "norm_quant.hip", "swiglu_quant.hip", "gemm.hip", "gemm_w4.hip", "gemm_skinny.hip",
           "gemm_stream.hip", "gemm_stream_e4m3_tiled.hip", "gemm_stream_e4m3_rows.hip", "gemm_stream_int8_tiled.hip",
           "gemm_stream_int8_rows.hip", "capi.hip"]

# Native tensor wrappers (host code against torch's C++ interface), linked to LIB.
TORCH_SRC = "torch_ops.cpp"
TORCH_LIB = PKG / "_h3q_torch.so"

HIPCC_FLAGS = [
    "--offload-arch=gfx950",
    "-O3",
    "-std=c++17",
    "-fPIC",
    "-fvisibility=hidden",
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wall",
]


def hipcc() -> str:
    for cand in (os.environ.get("HIPCC"), "/opt/rocm/bin/hipcc", shutil.which("hipcc")):
        if cand and Path(cand).exists():
            return cand
    raise RuntimeError("hipcc not found (ROCm is required to build the gfx950 library)")


def _quiet(text: str) -> str:
    # hipcc's host pass does not know the GPU-only feature flag; drop that note.
    return "\n".join(l for l in text.splitlines() if "packed-fp32-ops" not in l)


def _compile(cc: str, src: str, obj: Path) -> subprocess.CompletedProcess:
    cmd = [cc, *HIPCC_FLAGS, "-c", str(CSRC / src), "-o", str(obj)]
    return subprocess.run(cmd, capture_output=True, text=True)


def build(verbose: bool = False) -> Path:
    objdir = PKG / "_build"
    objdir.mkdir(exist_ok=True)
    cc = hipcc()
    objects = [objdir / (src + ".o") for src in SOURCES]
    # One hipcc per source, at most as many at once as there are CPUs (8 here);
    # the GEMM instances take longest and go first.
    workers = max(1, min(len(SOURCES) + 1, os.cpu_count() or 1, 8))
    with ThreadPoolExecutor(max_workers=workers) as pool:
        slow_first = sorted(zip(SOURCES, objects), key=lambda so: not so[0].startswith("gemm"))
        torch_object = pool.submit(_compile_torch, objdir / (TORCH_SRC + ".o"))
        jobs = {src: pool.submit(_compile, cc, src, obj) for src, obj in slow_first}
        results = [jobs[src].result() for src in SOURCES]
        torch_result = torch_object.result()
    for src, res in zip(SOURCES, results):
        if res.returncode != 0:
            raise RuntimeError(f"hipcc failed on {src}:\n{_quiet(res.stderr)}")
        if verbose and _quiet(res.stderr).strip():
            print(_quiet(res.stderr), file=sys.stderr)
    _link(cc, [str(o) for o in objects], LIB)
    ceil_obj = objdir / (CEILINGS_SRC + ".o")
    res = _compile(cc, CEILINGS_SRC, ceil_obj)
    if res.returncode != 0:
        raise RuntimeError(f"hipcc failed on {CEILINGS_SRC}:\n{_quiet(res.stderr)}")
    _link(cc, [str(ceil_obj)], CEILINGS_LIB)
    if torch_result.returncode != 0:
        raise RuntimeError(f"g++ failed on {TORCH_SRC}:\n{torch_result.stderr}")
    _link_torch(objdir / (TORCH_SRC + ".o"))
    return LIB


def _compile_torch(obj: Path) -> subprocess.CompletedProcess:
    import torch
    from torch.utils import cpp_extension

    includes = [f"-I{path}" for path in (*cpp_extension.include_paths(), sysconfig.get_paths()["include"])]
    cmd = ["g++", "-O2", "-std=c++17", "-fPIC", "-fvisibility=hidden", "-w",
           f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}",
           f"-DTORCH_EXTENSION_NAME={TORCH_LIB.stem}", *includes, "-c", str(CSRC / TORCH_SRC), "-o", str(obj)]
    return subprocess.run(cmd, capture_output=True, text=True)


def _link_torch(obj: Path) -> None:
    from torch.utils import cpp_extension

    tmp = TORCH_LIB.with_suffix(".so.tmp")
    cmd = ["g++", "-shared", "-fPIC", "-o", str(tmp), str(obj), f"-L{cpp_extension.TORCH_LIB_PATH}", "-ltorch_python",
           "-ltorch", "-ltorch_cpu", "-lc10", f"-L{PKG}", f"-l:{LIB.name}", "-Wl,-rpath,$ORIGIN"]
    res = subprocess.run(cmd, capture_output=True, text=True)
    if res.returncode != 0:
        raise RuntimeError(f"link of {TORCH_LIB.name} failed:\n{res.stderr}")
    os.replace(tmp, TORCH_LIB)


def _link(cc: str, objects: list[str], out: Path) -> None:
    tmp = out.with_suffix(".so.tmp")
    cmd = [cc, "--offload-arch=gfx950", "-shared", "-fPIC", "-o", str(tmp), *objects]
    res = subprocess.run(cmd, capture_output=True, text=True)
    if res.returncode != 0:
        raise RuntimeError(f"link of {out.name} failed:\n{_quiet(res.stderr)}")
    os.replace(tmp, out)


if __name__ == "__main__":
    print(build(verbose=True))
