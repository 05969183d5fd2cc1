"""Compile the HIP sources in this directory into ``kvax_amd/libkvax_amd.so`` for gfx950.

Usage: ``python -m kvax_amd.csrc.build`` (or ``build()`` from Python; ``python kvax_amd/csrc/build.py`` where there is no
torch).  hipcc cross-compiles, so no GPU is needed.  The library is built in-tree next to the Python package, and with it,
where torch and g++ are there, the extension module ``kvax_amd/_host.so``.
"""
from __future__ import annotations

import os
import shutil
import subprocess
import sys
from concurrent.futures import ThreadPoolExecutor
from pathlib import Path

CSRC = Path(__file__).resolve().parent
PKG = CSRC.parent
ROOT = PKG.parent
LIB = PKG / "libkvax_amd.so"
OBJ = CSRC / "build"

HOST = PKG / "_host.so"  # host.cpp: the host side of the calls, a Python extension module

SOURCES = ["abi.cpp", "mask_builder.hip", "fa_tiles.hip", "permute.hip", "fa_fwd.hip", "fa_bwd.hip"]

HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
FLAGS = [
    "--offload-arch=gfx950", "-O3", "-std=c++17", "-fPIC",
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    # MFMA results go to ordinary vector registers (where the element-wise code reads them) also in
    # kernels that run one wavefront per SIMD and may use the accumulation registers as well
    "-mllvm", "-amdgpu-mfma-vgpr-form=1",
    "-Wno-unused-command-line-argument", "-Wno-unknown-warning-option",
    f"-I{ROOT / 'include'}", f"-I{CSRC}",
]


def _compile(src: str, extra: list[str]) -> Path:
    OBJ.mkdir(exist_ok=True)
    out = OBJ / (src + ".o")
    cmd = [HIPCC, *FLAGS, *extra, "-x", "hip", "-c", str(CSRC / src), "-o", str(out)]
    r = subprocess.run(cmd, capture_output=True, text=True)
    # hipcc's host pass warns that it does not know the packed-fp32 target feature: harmless
    err = "\n".join(l for l in r.stderr.splitlines() if "packed-fp32-ops" not in l)
    if r.returncode != 0:
        raise RuntimeError(f"hipcc failed on {src}:\n{err}")
    if err.strip():
        print(err, file=sys.stderr)
    return out


def _compile_host() -> Path | None:
    """The extension module ``kvax_amd._host``: plain C++ against torch's headers and libraries.  Nothing else needs them
    or g++: without them it is left out."""
    import sysconfig

    try:
        import torch
    except ImportError:
        torch = None
    if torch is None or not shutil.which("g++"):
        print(f"{HOST.name} is left out: no {'torch' if torch is None else 'g++'}", file=sys.stderr)
        return None
    root = Path(torch.__file__).resolve().parent
    cmd = ["g++", "-O2", "-std=c++17", "-fPIC", "-shared", f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}",
           f'-DKVAX_TORCH_VERSION="{torch.__version__}"',
           f"-I{ROOT / 'include'}", f"-isystem{root / 'include'}", f"-isystem{root / 'include/torch/csrc/api/include'}",
           f"-I{sysconfig.get_paths()['include']}", str(CSRC / "host.cpp"), "-o", str(HOST),
           f"-L{root / 'lib'}", "-ltorch_python", "-ltorch_cpu", "-lc10"]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"g++ failed on host.cpp:\n{r.stderr}")
    return HOST


def build(extra_flags: list[str] | None = None, jobs: int = 4, lib: Path | None = None) -> Path:
    """Compile and link; ``lib`` overrides the output path (used for experimental variants,
    loaded by pointing the KVAX_AMD_LIB environment variable at them)."""
    global LIB, OBJ
    if lib is not None:
        LIB = Path(lib).resolve()
        OBJ = LIB.parent / (LIB.stem + "_obj")
    extra = list(extra_flags or [])
    sources = [s for s in SOURCES if (CSRC / s).exists()]
    with ThreadPoolExecutor(max_workers=jobs) as ex:
        host = ex.submit(_compile_host) if lib is None else None
        objs = list(ex.map(lambda s: _compile(s, extra), sources))
        cmd = [HIPCC, "--offload-arch=gfx950", "-shared", "-fPIC", "-o", str(LIB), *map(str, objs)]
        r = subprocess.run(cmd, capture_output=True, text=True)
        if r.returncode != 0:
            raise RuntimeError(f"link failed:\n{r.stderr}")
        if host is not None:
            host.result()  # raises once the library is there, which does not need it
    return LIB


if __name__ == "__main__":
    args = sys.argv[1:]
    out = None
    if args and args[0] == "-o":
        out, args = Path(args[1]), args[2:]
    print(build(args, lib=out))
