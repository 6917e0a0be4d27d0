"""The optional native modules of the package (mlir_edsl_hip/build.py), on the CPU."""
from __future__ import annotations

import os
from types import SimpleNamespace

import pytest

torch = pytest.importorskip("torch")

from mlir_edsl_hip import build, device


@pytest.mark.parametrize("fault", ["no_compiler", "compiler_fails", "no_headers"])
def test_build_goes_on_without_the_torch_module(fault, monkeypatch, tmp_path):
    """The device API works without it: a warning, and no module of an earlier build."""
    monkeypatch.setattr(build, "PKG_DIR", str(tmp_path))
    stale = build._module_path("_torch_launch")
    with open(stale, "w") as f:
        f.write("stale")
    if fault == "no_headers":
        def refuse(*_):
            raise ImportError("no headers")
        import torch.utils.cpp_extension
        monkeypatch.setattr(torch.utils.cpp_extension, "include_paths", refuse)
    else:
        monkeypatch.setenv("CXX", "/nonexistent/c++" if fault == "no_compiler" else "false")
    with pytest.warns(UserWarning, match="operands in Python"):
        assert build.build_optional_torch_launch_module() == []
    assert not os.path.exists(stale)


def test_a_module_of_another_torch_is_not_used():
    device._torch_module()
    assert device._native_checks(torch) is not None, "the torch launch module is not built"
    for version, commit in ((torch.__version__ + "x", torch.version.git_version), (torch.__version__, "0" * 40)):
        other = SimpleNamespace(__version__=version, version=SimpleNamespace(git_version=commit))
        assert device._native_checks(other) is None
