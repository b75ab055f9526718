"""Build libmica_amd.so in-tree: every source under mica_amd/csrc compiled for gfx950 with hipcc; and _native.so,
the host-side launch path (mica_amd/binding), with g++ against torch's headers.

    python -m mica_amd.build [--jobs N]

Flags: -O3, no fast-math (the quantizer needs IEEE fp32 division and square root),
-ffp-contract=off (fp32 steps round where the reference's torch code rounds; intended FMAs are
written as explicit fma builtins), packed-fp32 instructions disabled.
"""
from __future__ import annotations

import argparse
import concurrent.futures as cf
import os
import shutil
import subprocess
import sys
from pathlib import Path

PKG = Path(__file__).resolve().parent
CSRC = PKG / "csrc"
OUT = PKG / "libmica_amd.so"
BINDING = PKG / "binding" / "native.cpp"
NATIVE = PKG / "_native.so"
OBJ = PKG / "_build"
ARCH = "gfx950"

FLAGS = [
    f"--offload-arch={ARCH}",
    "-O3",
    "-std=c++17",
    "-fPIC",
    "-ffp-contract=off",
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wno-unused-command-line-argument",
]


def hipcc() -> str:
    for cand in (os.environ.get("HIPCC"), shutil.which("hipcc"), "/opt/rocm/bin/hipcc"):
        if cand and Path(cand).exists():
            return cand
    raise RuntimeError("hipcc not found (ROCm is required to build mica_amd)")


def sources():
    return sorted(list(CSRC.glob("*.hip")) + list(CSRC.glob("*.cpp")))


def _compile(src: Path) -> Path:
    obj = OBJ / (src.stem + ".o")
    cmd = [hipcc(), *FLAGS, "-c", str(src), "-o", str(obj)]
    if src.suffix == ".cpp":
        cmd[1:1] = ["-x", "hip"]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"hipcc failed for {src.name}:\n{' '.join(cmd)}\n{r.stdout}\n{r.stderr}")
    return obj


def _run(cmd, what):
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"{what} failed:\n{' '.join(cmd)}\n{r.stdout}\n{r.stderr}")


def build_native() -> Path:
    """Compile the launch path into _native.so (a CPython module; it calls libmica_amd.so through the addresses
    _lib.load() gives it, so the two are linked only to torch and Python)."""
    import sysconfig

    import torch
    from torch.utils import cpp_extension as ext

    rocm = Path(hipcc()).resolve().parent.parent
    libs = ext.library_paths()
    tmp = NATIVE.with_suffix(".so.tmp")
    _run(["g++", "-O2", "-std=c++17", "-fPIC", "-shared", "-fvisibility=hidden", "-DUSE_ROCM=1",
          "-D__HIP_PLATFORM_AMD__=1", f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}",
          *[f"-I{p}" for p in (*ext.include_paths(), rocm / "include", sysconfig.get_paths()["include"])],
          str(BINDING), "-o", str(tmp), *[f"-L{p}" for p in libs], *[f"-Wl,-rpath,{p}" for p in libs],
          "-ltorch_python", "-ltorch_cpu", "-ltorch", "-lc10", "-lc10_hip"], "g++ for native.cpp")
    os.replace(tmp, NATIVE)
    return NATIVE


def build(jobs: int | None = None, verbose: bool = True) -> Path:
    """Compile every source (always; never trusts an existing library), link libmica_amd.so and _native.so."""
    OBJ.mkdir(exist_ok=True)
    srcs = sources()
    jobs = jobs or min(len(srcs), os.cpu_count() or 4)
    with cf.ThreadPoolExecutor(max_workers=jobs) as ex:
        native = ex.submit(build_native)
        objs = list(ex.map(_compile, srcs))
        native.result()
    tmp = OUT.with_suffix(".so.tmp")
    cmd = [hipcc(), f"--offload-arch={ARCH}", "-shared", "-fPIC", "-o", str(tmp), *map(str, objs)]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"link failed:\n{' '.join(cmd)}\n{r.stdout}\n{r.stderr}")
    os.replace(tmp, OUT)
    if verbose:
        print(f"built {OUT} from {len(srcs)} sources", file=sys.stderr)
    return OUT


def main(argv=None):
    ap = argparse.ArgumentParser(description=__doc__)
    ap.add_argument("--jobs", type=int, default=None)
    args = ap.parse_args(argv)
    build(args.jobs)


if __name__ == "__main__":
    main()
