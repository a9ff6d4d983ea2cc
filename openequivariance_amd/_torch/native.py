"""Loads ``_oeq_torch-*.so``, the torch ops over the C ABI (``csrc/oeq_torch.cpp``), and builds it where no built file
exists. There is no other implementation of the ops: without the library every call of one is an error."""

from __future__ import annotations

import importlib.machinery
import importlib.util
import os
import subprocess
import sys
import sysconfig
import threading
from pathlib import Path

import torch

from .. import runtime as rt

# The file is bound to the torch it was compiled against (its C++ interface changes between releases), to this Python
# and to the C ABI: what was built for others has another name and is not loaded.
_SO_PATH = rt._PKG_DIR / f"_oeq_torch-{torch.__version__}-{sys.implementation.cache_tag}-abi{rt.ABI_VERSION}.so"
_SRC_PATH = rt._PKG_DIR / "csrc" / "oeq_torch.cpp"
_lock = threading.Lock()
_module = None


def build_ops(verbose: bool = False) -> Path:
    """Compile csrc/oeq_torch.cpp (host code only) against the installed torch, next to liboeq_amd.so."""
    root = Path(torch.__file__).resolve().parent
    rocm = os.environ.get("ROCM_PATH", "/opt/rocm")
    tmp = _SO_PATH.with_name(f"{_SO_PATH.name}.tmp{os.getpid()}")
    cmd = ["g++", "-O2", "-std=c++17", "-fPIC", "-shared", "-D__HIP_PLATFORM_AMD__=1", "-DUSE_ROCM=1",
           f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}",
           f"-I{rt._INCLUDE_DIR}", f"-I{root / 'include'}", f"-I{root / 'include/torch/csrc/api/include'}",
           f"-I{rocm}/include", f"-I{sysconfig.get_paths()['include']}", str(_SRC_PATH), "-o", str(tmp),
           f"-L{rt._PKG_DIR}", "-loeq_amd", f"-L{root / 'lib'}", "-ltorch", "-ltorch_cpu", "-ltorch_python", "-lc10",
           "-ltorch_hip", "-lc10_hip", "-Wl,-rpath,$ORIGIN"]
    res = subprocess.run(cmd, capture_output=True, text=True)
    if res.returncode != 0:
        tmp.unlink(missing_ok=True)
        raise rt.OeqError(f"building {_SO_PATH.name} failed:\n{res.stdout}\n{res.stderr}")
    os.replace(tmp, _SO_PATH)
    if verbose:
        print(" ".join(cmd).replace(str(tmp), str(_SO_PATH)))
    return _SO_PATH


def _stale() -> bool:
    built = _SO_PATH.stat().st_mtime
    return any(src.exists() and src.stat().st_mtime > built for src in (_SRC_PATH, rt._INCLUDE_DIR / "oeq_amd.h"))


def so_path() -> Path:
    return _SO_PATH


def load():
    """The extension module; loading it registers the ops ``torch.ops.oeq_amd.*``."""
    global _module
    with _lock:
        if _module is None:
            rt.load_library()  # (built if need be, bound to the HIP libraries torch has loaded, ABI checked)
            if not _SO_PATH.exists() or _stale():
                build_ops()
            loader = importlib.machinery.ExtensionFileLoader("_oeq_torch", str(_SO_PATH))
            spec = importlib.util.spec_from_file_location("_oeq_torch", str(_SO_PATH), loader=loader)
            module = importlib.util.module_from_spec(spec)
            loader.exec_module(module)
            if module.abi_version() != rt.ABI_VERSION:
                raise rt.OeqError(f"{_SO_PATH} was compiled for C ABI {module.abi_version()}, this package has "
                                  f"{rt.ABI_VERSION}: rebuild it")
            _module = module
    return _module
