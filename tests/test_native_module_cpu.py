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
