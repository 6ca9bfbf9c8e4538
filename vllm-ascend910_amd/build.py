"""Build recipe for the gfx950 HIP library behind the C ABI (include/w4a8_amd.h)
and for the torch op kernels over it.

Compiles every ``csrc/*.hip`` with hipcc for gfx950 only and links them into
``_lib/libw4a8_amd.so`` inside this package, and ``csrc/torch_ops.cpp`` (host code
only) with g++ into ``_lib/w4a8_torch.so``, so the built libraries travel with
the source tree.  Every call recompiles (kernel headers are real dependencies;
a stale library is never reused).

    python vllm-ascend910_amd/build.py        # or __graft_entry__.build()
"""
from __future__ import annotations

import concurrent.futures as cf
import os
import shutil
import subprocess
import sys
import sysconfig
from pathlib import Path

PKG = Path(__file__).resolve().parent
CSRC = PKG / "csrc"
LIBDIR = PKG / "_lib"
LIBNAME = "libw4a8_amd.so"
TORCH_LIBNAME = "w4a8_torch.so"   # imported as module w4a8_torch
ARCH = "gfx950"

# Packed-FP32 VALU forms are disabled for all device code on this platform;
# hipcc's host pass warns that it does not know the feature, which is harmless.
# MFMA results stay in ordinary VGPRs: the folds read every accumulator with
# VALU instructions, which cannot address AGPRs (each element would first need
# a v_accvgpr_read).
DEVICE_FLAGS = ["-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
                "-mllvm", "-amdgpu-mfma-vgpr-form=1"]
COMMON_FLAGS = ["-O3", "-std=c++17", "-fPIC", f"--offload-arch={ARCH}", "-Wall",
                "-Wno-unused-function", "-Wno-unused-variable"]


def hipcc() -> str:
    exe = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not os.path.exists(exe):
        raise FileNotFoundError("hipcc not found; the W4A8 library needs ROCm's hipcc")
    return exe


def _compile(src: Path, obj: Path) -> None:
    cmd = [hipcc(), *COMMON_FLAGS, *DEVICE_FLAGS, "-c", str(src), "-o", str(obj)]
    res = subprocess.run(cmd, capture_output=True, text=True)
    # Filter the known host-pass warning about the packed-fp32 feature.
    err = "\n".join(l for l in res.stderr.splitlines() if "packed-fp32-ops" not in l)
    if res.returncode != 0:
        raise RuntimeError(f"hipcc failed for {src.name}:\n{err}")
    if err.strip():
        sys.stderr.write(err + "\n")


def build_torch(verbose: bool = False) -> Path:
    """Compile csrc/torch_ops.cpp against the torch of this interpreter; returns its path."""
    import torch
    root = Path(torch.__file__).resolve().parent
    rocm = Path(hipcc()).resolve().parents[1]
    LIBDIR.mkdir(exist_ok=True)
    out, tmp = LIBDIR / TORCH_LIBNAME, LIBDIR / (TORCH_LIBNAME + ".tmp")
    cmd = [shutil.which("g++") or "g++", "-O2", "-std=c++17", "-fPIC", "-shared", "-fvisibility=hidden",
           f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}", "-DUSE_ROCM=1",
           "-DTORCH_EXTENSION_NAME=w4a8_torch",
           *(f"-isystem{d}" for d in (root / "include", root / "include" / "torch" / "csrc" / "api" / "include",
                                      rocm / "include", sysconfig.get_paths()["include"])),
           str(CSRC / "torch_ops.cpp"), "-o", str(tmp), f"-L{root / 'lib'}", "-ltorch", "-ltorch_cpu",
           "-ltorch_python", "-lc10", "-lc10_hip"]
    res = subprocess.run(cmd, capture_output=True, text=True)
    if res.returncode != 0:
        raise RuntimeError(f"g++ failed for torch_ops.cpp:\n{res.stderr}")
    os.replace(tmp, out)
    if verbose:
        print(f"built {out}")
    return out


def build(verbose: bool = False, jobs: int = 8) -> Path:
    """Compile and link both libraries; returns the HIP library's path."""
    objdir = PKG / "_build"
    objdir.mkdir(exist_ok=True)
    LIBDIR.mkdir(exist_ok=True)
    srcs = sorted(CSRC.glob("*.hip"))
    objs = [objdir / (s.stem + ".o") for s in srcs]
    with cf.ThreadPoolExecutor(max_workers=max(1, min(jobs, len(srcs)))) as ex:
        native = ex.submit(build_torch, verbose)
        list(ex.map(lambda so: _compile(*so), zip(srcs, objs)))
        native.result()
    out = LIBDIR / LIBNAME
    tmp = LIBDIR / (LIBNAME + ".tmp")
    cmd = [hipcc(), f"--offload-arch={ARCH}", "-shared", "-fPIC", "-o", str(tmp), *map(str, objs)]
    res = subprocess.run(cmd, capture_output=True, text=True)
    if res.returncode != 0:
        raise RuntimeError(f"link failed:\n{res.stderr}")
    # A kernel whose host launch stub the compiler dropped links fine and
    # fails only when the library is loaded: refuse such a build here.
    nm = shutil.which("nm")
    if nm:
        syms = subprocess.run([nm, "-D", "--undefined-only", str(tmp)], capture_output=True, text=True).stdout
        missing = [l.split()[-1] for l in syms.splitlines() if "__device_stub__" in l]
        if missing:
            raise RuntimeError(f"undefined kernel launch stubs in {tmp.name}: {missing[:4]}")
    os.replace(tmp, out)
    if verbose:
        print(f"built {out}")
    return out


if __name__ == "__main__":
    build(verbose=True)
