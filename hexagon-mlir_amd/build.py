"""Build libhxmi.so (the C-ABI kernel library) in-tree with hipcc for gfx950,
and hxmi_torch.so (the native entry of the torch-facing ops) on top of it
where torch and its headers are there.

    python hexagon-mlir_amd/build.py [--jobs N]

Every ``csrc/*.hip`` is compiled to an object in ``csrc/_build/`` in
parallel, then linked into ``lib/libhxmi.so``.  The build always recompiles
(it is the "does it build" check); it needs hipcc but no GPU.
"""
from __future__ import annotations

import argparse
import concurrent.futures as cf
import os
import pathlib
import shutil
import subprocess
import sys

PKG = pathlib.Path(__file__).resolve().parent
CSRC = PKG / "csrc"
BUILD = CSRC / "_build"
LIB = PKG / "lib" / "libhxmi.so"
OPS = PKG / "lib" / "hxmi_torch.so"
ARCH = "gfx950"

# -packed-fp32-ops: keep hipcc from emitting packed fp32 VALU ops.
HIPFLAGS = [
    f"--offload-arch={ARCH}",
    "-O3",
    "-std=c++17",
    "-fPIC",
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wno-unused-command-line-argument",
]


# Per-source extra flags.  The attention kernel rescales its MFMA accumulators
# with vector ALU ops between MFMAs; with accumulators in AGPRs (the
# compiler's default) every key block copies them to VGPRs and back, so its
# files ask for the VGPR form of the MFMA operands.
EXTRA = {f"attention_{t}.hip": ["-mllvm", "-amdgpu-mfma-vgpr-form"] for t in ("f16", "bf16")}


def hipcc() -> str:
    for cand in (os.environ.get("HIPCC"), "/opt/rocm/bin/hipcc", shutil.which("hipcc")):
        if cand and os.path.exists(cand):
            return cand
    raise RuntimeError("hipcc not found (ROCm is required to build libhxmi.so)")


def _compile(src: pathlib.Path) -> pathlib.Path:
    obj = BUILD / (src.stem + ".o")
    cmd = [hipcc(), *HIPFLAGS, *EXTRA.get(src.name, []), "-c", str(src), "-o", str(obj)]
    proc = subprocess.run(cmd, capture_output=True, text=True)
    if proc.returncode != 0:
        raise RuntimeError(f"compile failed: {' '.join(cmd)}\n{proc.stdout}\n{proc.stderr}")
    return obj


def _build_ops() -> None:
    """torch_ops.cpp is host code only: g++ against torch's headers, linked to
    the libhxmi.so beside it."""
    OPS.unlink(missing_ok=True)  # (one of another libhxmi.so)
    import sysconfig

    import torch
    from torch.utils import cpp_extension

    root = pathlib.Path(torch.__file__).parent
    inc = [*cpp_extension.include_paths(), sysconfig.get_paths()["include"], "/opt/rocm/include"]
    tmp = OPS.with_suffix(".so.tmp")
    cmd = ["g++", "-O2", "-std=c++17", "-fPIC", "-shared", "-DUSE_ROCM=1", "-D__HIP_PLATFORM_AMD__=1",
           f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}", *(f"-I{p}" for p in inc),
           str(CSRC / "torch_ops.cpp"), "-o", str(tmp), f"-L{root / 'lib'}", "-lc10", "-lc10_hip", "-ltorch_cpu",
           "-ltorch_python", f"-L{LIB.parent}", "-lhxmi", "-Wl,-rpath,$ORIGIN"]
    proc = subprocess.run(cmd, capture_output=True, text=True)
    if proc.returncode != 0:
        raise RuntimeError(f"compile failed: {' '.join(cmd)}\n{proc.stdout}\n{proc.stderr}")
    os.replace(tmp, OPS)


def build_ops() -> bool:
    """hxmi_torch.so, or False with the reason on stderr: libhxmi.so and the
    ops work without it (no torch or no ROCm torch headers here)."""
    try:
        _build_ops()
    except (ImportError, OSError, RuntimeError) as e:
        print(f"[hxmi] {OPS.name} is not built, the ops take their Python forms: {e}", file=sys.stderr, flush=True)
        return False
    return True


def build(jobs: int | None = None, verbose: bool = True) -> pathlib.Path:
    BUILD.mkdir(parents=True, exist_ok=True)
    LIB.parent.mkdir(parents=True, exist_ok=True)
    sources = sorted(CSRC.glob("*.hip"))
    jobs = jobs or min(len(sources), os.cpu_count() or 4, 16)
    if verbose:
        print(f"[hxmi] compiling {len(sources)} sources for {ARCH} with {jobs} jobs", flush=True)
    with cf.ThreadPoolExecutor(max_workers=jobs) as ex:
        objs = list(ex.map(_compile, sources))
    tmp = LIB.with_suffix(".so.tmp")
    cmd = [hipcc(), f"--offload-arch={ARCH}", "-shared", "-fPIC", "-o", str(tmp), *map(str, objs)]
    proc = subprocess.run(cmd, capture_output=True, text=True)
    if proc.returncode != 0:
        raise RuntimeError(f"link failed: {' '.join(cmd)}\n{proc.stdout}\n{proc.stderr}")
    os.replace(tmp, LIB)
    built_ops = build_ops()
    if verbose:
        print(f"[hxmi] built {LIB}" + (f" and {OPS.name}" if built_ops else ""), flush=True)
    return LIB


if __name__ == "__main__":
    ap = argparse.ArgumentParser()
    ap.add_argument("--jobs", type=int, default=None)
    args = ap.parse_args()
    build(args.jobs)
    sys.exit(0)
