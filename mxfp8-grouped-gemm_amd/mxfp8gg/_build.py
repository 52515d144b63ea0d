"""Build libmxgg.so (gfx950 HIP kernels + C ABI) in-tree with hipcc, and the host
module _mxgg_host.so (csrc/host.cpp) with g++.

The shared library lands next to this file so that it travels with the
source tree; nothing is installed into site-packages.
"""
from __future__ import annotations

import concurrent.futures as _cf
import os
import shutil
import subprocess
from pathlib import Path

PKG_DIR = Path(__file__).resolve().parent
CSRC_DIR = PKG_DIR.parent / "csrc"
INCLUDE_DIR = PKG_DIR.parent.parent / "include"
BUILD_DIR = PKG_DIR.parent / "_build"
LIB_PATH = PKG_DIR / "libmxgg.so"
HOST_PATH = PKG_DIR / "_mxgg_host.so"

SOURCES = ["capi.hip", "quant.hip", "swiglu.hip", "route.hip", "groups.hip", "gemm.hip"]
HEADERS = ["mxgg_internal.h", "mx_device.h", "gemm_thin.h", "wgrad_ahead.h"]

ARCH = os.environ.get("MXGG_OFFLOAD_ARCH", "gfx950")

# -packed-fp32-ops: keep v_pk_{add,mul,fma}_f32 out of the generated code.
HIPCC_FLAGS = [
    f"--offload-arch={ARCH}",
    "-O3",
    "-fPIC",
    "-std=c++17",
    "-Wall",
    "-Wno-unused-function",
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    f"-I{INCLUDE_DIR}",
]


def hipcc() -> str:
    cand = os.environ.get("HIPCC") or shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    return cand


def _run(cmd: list[str]) -> None:
    proc = subprocess.run(cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
    # hipcc's host pass does not know the packed-fp32 feature and says so; drop that line.
    out = "\n".join(
        ln for ln in proc.stdout.splitlines()
        if "packed-fp32-ops" not in ln and "--hip-link" not in ln
    )
    if proc.returncode != 0:
        raise RuntimeError(f"command failed ({proc.returncode}): {' '.join(cmd)}\n{out}")
    if out.strip():
        print(out)


def _host_command(out: Path) -> list[str]:
    """g++ command of the host module (csrc/host.cpp, a torch extension without device code)."""
    import sysconfig

    import torch
    from torch.utils import cpp_extension

    includes = [*cpp_extension.include_paths(), sysconfig.get_paths()["include"]]
    libdirs = cpp_extension.library_paths()
    return [
        os.environ.get("CXX") or shutil.which("g++") or "g++", "-O2", "-std=c++17", "-fPIC",
        "-shared", "-fvisibility=hidden", "-DTORCH_API_INCLUDE_EXTENSION_H",
        f"-DTORCH_EXTENSION_NAME={HOST_PATH.name.split('.')[0]}",
        f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}",
        *[f"-isystem{d}" for d in includes], str(CSRC_DIR / "host.cpp"), "-o", str(out),
        *[f"-L{d}" for d in libdirs], "-lc10", "-ltorch_cpu", "-ltorch", "-ltorch_python",
    ]


def build(verbose: bool = True) -> Path:
    """Compile every HIP source for gfx950, link libmxgg.so and build the host
    module beside it (always rebuilds).  The library is in place also where
    the host module does not build, which is raised last."""
    BUILD_DIR.mkdir(parents=True, exist_ok=True)
    cc = hipcc()
    objs = []
    cmds = []
    for src in SOURCES:
        obj = BUILD_DIR / (Path(src).stem + ".o")
        objs.append(obj)
        cmds.append([cc, *HIPCC_FLAGS, "-c", str(CSRC_DIR / src), "-o", str(obj)])
    host_tmp = HOST_PATH.with_suffix(".so.tmp")
    with _cf.ThreadPoolExecutor(max_workers=len(cmds) + 1) as ex:
        host = ex.submit(lambda: _run(_host_command(host_tmp)))
        list(ex.map(_run, cmds))
        tmp = LIB_PATH.with_suffix(".so.tmp")
        _run([cc, "-shared", "-fPIC", f"--offload-arch={ARCH}", *map(str, objs), "-o", str(tmp)])
        os.replace(tmp, LIB_PATH)
        host.result()
    os.replace(host_tmp, HOST_PATH)
    if verbose:
        print(f"[mxfp8gg] built {LIB_PATH}")
    return LIB_PATH


if __name__ == "__main__":
    build()
