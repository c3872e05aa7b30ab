"""Builds libdeca_hip.so (the C-ABI loader/launcher) in-tree with hipcc, and `_launch`, the extension
module through which a loaded kernel is called with torch tensors."""

from __future__ import annotations

import os
import subprocess
import sysconfig

PKG_ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
REPO_ROOT = os.path.dirname(PKG_ROOT)
LIB_PATH = os.path.join(PKG_ROOT, "libdeca_hip.so")
SOURCE = os.path.join(PKG_ROOT, "csrc", "deca_hip.cpp")
# (named for the interpreter it is built for: no other one takes it)
EXT_PATH = os.path.join(PKG_ROOT, "_launch" + sysconfig.get_config_var("EXT_SUFFIX"))
EXT_SOURCE = os.path.join(PKG_ROOT, "csrc", "launch_ext.cpp")
INCLUDE_DIR = os.path.join(REPO_ROOT, "include")


def build_library(force: bool = True) -> str:
    if not force and os.path.exists(LIB_PATH):
        return LIB_PATH
    from deca_amd.kernels.build import hipcc_path

    tmp = f"{LIB_PATH}.tmp{os.getpid()}"
    cmd = [
        hipcc_path(), "-O2", "-std=c++17", "-fPIC", "-shared", f"-I{INCLUDE_DIR}",
        SOURCE, "-o", tmp,
    ]
    proc = subprocess.run(cmd, capture_output=True, text=True)
    if proc.returncode != 0:
        raise RuntimeError(f"building libdeca_hip.so failed:\n{proc.stderr[-4000:]}")
    os.replace(tmp, LIB_PATH)
    return LIB_PATH


def build_extension(force: bool = True) -> str:
    """`_launch` against the headers and libraries of the torch it will run with (host code
    only); links the launcher library beside it."""
    if not force and os.path.exists(EXT_PATH):
        return EXT_PATH
    import torch
    from torch.utils import cpp_extension

    tmp = f"{EXT_PATH}.tmp{os.getpid()}"
    includes = [INCLUDE_DIR, sysconfig.get_paths()["include"], *cpp_extension.include_paths("cuda")]
    cmd = [
        "g++", "-O2", "-std=c++17", "-fPIC", "-shared", "-D__HIP_PLATFORM_AMD__=1", "-DUSE_ROCM=1",
        f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}",
        f'-DDECA_TORCH="{torch.__version__}"', *(f"-I{d}" for d in includes),
        EXT_SOURCE, "-o", tmp, f"-L{os.path.join(os.path.dirname(torch.__file__), 'lib')}",
        "-lc10", "-lc10_hip", "-ltorch_cpu", "-ltorch_python",
        f"-L{PKG_ROOT}", f"-l:{os.path.basename(LIB_PATH)}", "-Wl,-rpath,$ORIGIN",
    ]
    proc = subprocess.run(cmd, capture_output=True, text=True)
    if proc.returncode != 0:
        raise RuntimeError(f"building {os.path.basename(EXT_PATH)} failed:\n{proc.stderr[-4000:]}")
    os.replace(tmp, EXT_PATH)
    return EXT_PATH


if __name__ == "__main__":
    print(build_library())
    print(build_extension())
