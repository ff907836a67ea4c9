"""Build recipe for the gfx950 HIP library ``fna2_amd/libfna2_hip.so`` and
its torch binding ``fna2_amd/_torch_binding.so``.

Every HIP source in ``fna2_amd/csrc`` is compiled by ``hipcc`` for gfx950 only
and linked into one shared library that exports the C ABI of
``include/fna2.h``.  ``fna2_torch.cpp`` (host code: the launch path of the
Python entry points) is compiled by the same ``hipcc`` against torch's headers.
Objects go to ``fna2_amd/_build`` (git-ignored); the library is written in-tree
so that it travels with the source tree.

Run as ``python -m fna2_amd.build``.
"""
from __future__ import annotations

import concurrent.futures
import os
import shutil
import subprocess
import sys
from pathlib import Path

PKG = Path(__file__).resolve().parent
ROOT = PKG.parent
CSRC = PKG / "csrc"
BUILD = PKG / "_build"
LIB = PKG / "libfna2_hip.so"
BINDING = PKG / "_torch_binding.so"

ARCH = "gfx950"
HIPCC = os.environ.get("HIPCC", shutil.which("hipcc") or "/opt/rocm/bin/hipcc")

# Packed FP32 (v_pk_*_f32) is switched off for all device code.
COMMON = [
    f"--offload-arch={ARCH}",
    "-O3",
    "-std=c++17",
    "-fPIC",
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    f"-I{ROOT / 'include'}",
    f"-I{CSRC}",
]

SOURCES = ["fna2_capi.cpp", "fna2_sched.hip", "fna2_fwd.hip", "fna2_bwd.hip", "fna2_bwd_dkdv.hip",
           "fna2_bwd_dq.hip", "fna2_rope.hip", "fna2_decode.hip"]


def _compile(src: Path, obj: Path, verbose: bool) -> None:
    cmd = [HIPCC, *COMMON, "-c", str(src), "-o", str(obj)]
    if src.suffix == ".cpp":
        cmd[1:1] = ["-x", "hip"]
    if verbose:
        print(" ".join(cmd), flush=True)
    res = subprocess.run(cmd, capture_output=True, text=True)
    # hipcc's host pass does not know the packed-fp32 feature: drop that note.
    noise = "'-packed-fp32-ops' is not a recognized feature"
    err = "\n".join(l for l in res.stderr.splitlines() if noise not in l)
    if res.returncode != 0:
        raise RuntimeError(f"hipcc failed on {src.name}:\n{err}")
    if verbose and err.strip():
        print(err, file=sys.stderr)


def _build_binding(verbose: bool) -> None:
    """fna2_torch.cpp -> _torch_binding.so (a Python extension module)."""
    import sysconfig

    import torch
    from torch.utils import cpp_extension

    inc = [*cpp_extension.include_paths(), sysconfig.get_path("include"), "/opt/rocm/include",
           str(ROOT / "include")]
    libdir = cpp_extension.library_paths()[0]
    tmp = BINDING.with_suffix(".so.tmp")
    cmd = [HIPCC, "-x", "c++", "-O2", "-std=c++17", "-fPIC", "-shared", "-D__HIP_PLATFORM_AMD__=1",
           "-DUSE_ROCM=1", f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}",
           "-DTORCH_EXTENSION_NAME=_torch_binding", "-DTORCH_API_INCLUDE_EXTENSION_H", "-w",
           *[a for d in inc for a in ("-isystem", d)], str(CSRC / "fna2_torch.cpp"), "-o", str(tmp),
           f"-L{libdir}", "-lc10", "-lc10_hip", "-ltorch_cpu", "-ltorch", "-ltorch_python"]
    if verbose:
        print(" ".join(cmd), flush=True)
    res = subprocess.run(cmd, capture_output=True, text=True)
    if res.returncode != 0:
        raise RuntimeError(f"hipcc failed on fna2_torch.cpp:\n{res.stderr}")
    os.replace(tmp, BINDING)


def build(verbose: bool = False, jobs: int = 5) -> Path:
    """Compile all HIP sources for gfx950 and link ``libfna2_hip.so``; build
    the torch binding."""
    BUILD.mkdir(exist_ok=True)
    srcs = [CSRC / s for s in SOURCES]
    objs = [BUILD / (s.stem + ".o") for s in srcs]
    with concurrent.futures.ThreadPoolExecutor(max_workers=jobs) as ex:
        futs = [ex.submit(_build_binding, verbose)]
        futs += [ex.submit(_compile, s, o, verbose) for s, o in zip(srcs, objs)]
        for f in futs:
            f.result()
    tmp = LIB.with_suffix(".so.tmp")
    cmd = [HIPCC, f"--offload-arch={ARCH}", "-shared", "-fPIC", "-o", str(tmp), *map(str, objs)]
    if verbose:
        print(" ".join(cmd), flush=True)
    res = subprocess.run(cmd, capture_output=True, text=True)
    if res.returncode != 0:
        raise RuntimeError(f"link failed:\n{res.stderr}")
    # The library must load (an unresolved host symbol would only show at dlopen).
    chk = subprocess.run([sys.executable, "-c", f"import ctypes; ctypes.CDLL({str(tmp)!r})"],
                         capture_output=True, text=True)
    if chk.returncode != 0:
        raise RuntimeError(f"built library does not load:\n{chk.stderr.strip()}")
    os.replace(tmp, LIB)
    return LIB


if __name__ == "__main__":
    print(build(verbose="-v" in sys.argv))
