"""The extension module of csrc/host.cpp is needed by the attention types with a plain cache and by nothing else."""
import sys

import pytest

import infllm_amd
from infllm_amd import _lib


@pytest.fixture
def fresh(monkeypatch):
    """nothing loaded yet"""
    monkeypatch.setattr(_lib, "_lib", None)
    monkeypatch.setattr(_lib, "_host", None)
    return monkeypatch


def test_the_library_loads_without_it(fresh):
    fresh.delattr(infllm_amd, "_host", raising=False)
    fresh.setitem(sys.modules, "infllm_amd._host", None)               # (an import of it fails)
    assert _lib.load().infllm_version() == _lib.ABI_VERSION
    with pytest.raises(_lib.InfLLMHipError, match="_host"):
        _lib.host()


def test_it_is_given_the_library_that_is_loaded(fresh):
    seen = []

    class Module:
        bind = staticmethod(lambda *a: seen.append(a))
    fresh.setattr(infllm_amd, "_host", Module, raising=False)
    for _ in range(2):                                                 # (a library that is loaded anew has functions of its own)
        fresh.setattr(_lib, "_lib", None)
        lib = _lib.load()
        assert _lib.host() is Module and _lib.host() is Module
        assert seen.pop()[0] is lib.infllm_window_forward and not seen
