"""Building and importing the package from states that a working tree can be in."""

import os
import shutil
import subprocess
import sys
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parent.parent


@pytest.fixture
def tree(tmp_path):
    """A copy of the package's sources without anything built."""
    for name in ("openequivariance_amd", "include"):
        shutil.copytree(ROOT / name, tmp_path / name,
                        ignore=shutil.ignore_patterns("*.so", "*.so.tmp*", "_kcache", "__pycache__"))
    shutil.copy(ROOT / "__graft_entry__.py", tmp_path)
    return tmp_path


def _python(tree, code, **env):
    return subprocess.run([sys.executable, "-c", code], cwd=tree, capture_output=True, text=True,
                          env=dict(os.environ, PYTHONPATH=str(tree), **env))


def test_build_replaces_a_library_of_another_abi(tree):
    lib = tree / "openequivariance_amd" / "liboeq_amd.so"
    (tree / "old.c").write_text("int oeq_abi_version(void) { return 6; }\n")
    subprocess.run(["gcc", "-shared", "-fPIC", str(tree / "old.c"), "-o", str(lib)], check=True)
    res = _python(tree, "import __graft_entry__ as g\n"
                        "rt = g.build_libraries()\n"
                        "print(rt.load_library().oeq_abi_version() == rt.ABI_VERSION)")
    assert res.returncode == 0, res.stderr
    assert res.stdout.split()[-1] == "True"


def test_import_needs_neither_built_libraries_nor_compilers(tree):
    """Problems and modules can be made with torch alone, meta tensors traced; a call of an op says what is missing."""
    (tree / "none").mkdir()
    res = _python(tree, """
import torch
import openequivariance_amd as oeq
from openequivariance_amd._torch import ops
p = oeq.TPProblem("4x1e", "1x1e", "4x0e", [(0, 0, 0, "uvu", True)], shared_weights=False, internal_weights=False)
tp = oeq.TensorProduct(p)
x, y, w = (torch.empty(3, n, device="meta") for n in (12, 3, 4))
assert ops.tp_forward(x, y, w, tp.kid).shape == (3, 4)
try:
    torch.ops.oeq_amd.tp_forward.default.redispatch(torch._C.DispatchKeySet(torch._C.DispatchKey.CUDA), x, y, w, tp.kid)
except oeq.runtime.OeqError as exc:
    assert "could not be loaded" in str(exc) and "hipcc" in str(exc), exc
    print("refused")
""", PATH=str(tree / "none"))
    assert res.returncode == 0, res.stderr
    assert res.stdout.split()[-1] == "refused"


def test_ops_built_for_another_torch_are_not_loaded(tree):
    from openequivariance_amd import runtime as rt
    from openequivariance_amd._torch import native
    assert native.load().abi_version() == rt.ABI_VERSION
    pkg = tree / "openequivariance_amd"
    shutil.copy(rt.lib_path(), pkg)
    built = native.so_path()
    for other in ("_oeq_torch.so", built.name.replace("torch-", "torch-1."), built.name.replace("-abi", "-abi1")):
        shutil.copy(built, pkg / other)
    (tree / "none").mkdir()
    code = "from openequivariance_amd._torch import ops; print(ops._native is None)"
    assert _python(tree, code, PATH=str(tree / "none")).stdout.split() == ["True"]
    shutil.copy(built, pkg)
    assert _python(tree, code, PATH=str(tree / "none")).stdout.split() == ["False"]
