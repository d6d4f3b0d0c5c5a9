"""The module that makes the plain call from native code: an extra that the library does without."""
import importlib.util
import os
import warnings

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PKG = os.path.join(ROOT, "ring-sliding-window-attention_amd")


@pytest.fixture
def fresh(monkeypatch):
    """ring_swa._lib as before the module is first asked for."""
    import __graft_entry__

    __graft_entry__.ensure_built()
    from ring_swa import _lib

    _lib.lib()
    monkeypatch.setattr(_lib, "_torch_calls", None)
    monkeypatch.delenv("RSWA_LIBRARY", raising=False)
    return _lib


def test_the_built_module_is_taken(fresh):
    with warnings.catch_warnings():
        warnings.simplefilter("error")
        assert fresh.torch_calls().params_bytes() > 0


def test_a_library_without_the_module_is_enough(fresh, monkeypatch, tmp_path):
    monkeypatch.setattr(fresh, "_PKG_ROOT", str(tmp_path))
    with pytest.warns(RuntimeWarning, match="missing"):
        assert fresh.torch_calls() is None
    with warnings.catch_warnings():  # (said once)
        warnings.simplefilter("error")
        assert fresh.torch_calls() is None


def test_a_module_of_another_pytorch_is_not_used(fresh, monkeypatch):
    """Its inlined accessors would read tensors at that PyTorch's layout."""
    monkeypatch.setattr(fresh, "torch_build", lambda: "another")
    with pytest.warns(RuntimeWarning, match="this is another"):
        assert fresh.torch_calls() is None


def test_a_module_that_does_not_load_is_not_used(fresh, monkeypatch, tmp_path):
    (tmp_path / "lib").mkdir()
    (tmp_path / "lib" / "rswa_torch.so").write_bytes(b"not a shared object")
    monkeypatch.setattr(fresh, "_PKG_ROOT", str(tmp_path))
    with pytest.warns(RuntimeWarning, match="another PyTorch"):
        assert fresh.torch_calls() is None


def test_another_pytorch_makes_the_build_stale(monkeypatch, tmp_path):
    spec = importlib.util.spec_from_file_location("rswa_build", os.path.join(PKG, "build.py"))
    build = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(build)
    runs = []

    def compiler(cmd, **kw):
        runs.append(cmd)
        open(cmd[cmd.index("-o") + 1], "w").close()
        return type("Result", (), dict(returncode=0, stdout="", stderr=""))

    monkeypatch.setattr(build.subprocess, "run", compiler)
    monkeypatch.setattr(build, "OBJ", str(tmp_path))
    monkeypatch.setattr(build, "LIBDIR", str(tmp_path))
    for _ in range(2):
        build._build_torch_calls(False)
    assert len(runs) == 1
    monkeypatch.setattr(build, "_torch_build", lambda: "another")
    for _ in range(2):
        build._build_torch_calls(False)
    assert len(runs) == 2 and '-DRSWA_TORCH_BUILD="another"' in runs[1]
