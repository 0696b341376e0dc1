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


def test_a_module_of_another_build_is_refused(fresh):
    import torch
    module, lib, block = _lib.host(), _lib.load(), _lib.C.sizeof(_lib.WindowArgs)
    told = [lib.infllm_window_forward, 1, _lib.ABI_VERSION, block, torch.__version__]
    for i, other in ((2, _lib.ABI_VERSION + 1), (3, block + 8), (4, torch.__version__ + "1")):
        with pytest.raises(ImportError, match="built"):
            module.bind(*told[:i], other, *told[i + 1:])
    fresh.setattr(_lib, "_host", None)
    with fresh.context() as m:                                         # a header that has moved on
        m.setattr(_lib, "ABI_VERSION", _lib.ABI_VERSION + 1)
        with pytest.raises(_lib.InfLLMHipError, match="_host.*built"):
            _lib.host()

    class Older:
        bind = staticmethod(lambda function, address: None)
    with fresh.context() as m:
        m.setattr(infllm_amd, "_host", Older)
        with pytest.raises(_lib.InfLLMHipError, match="_host"):
            _lib.host()
    assert _lib.host() is module


@pytest.mark.parametrize("broken", ["libinfllm_hip", "_host"])
def test_a_build_that_fails_leaves_both_as_they_were(broken, tmp_path, monkeypatch):
    from infllm_amd import build
    lib, host = tmp_path / "libinfllm_hip.so", tmp_path / "_host.so"
    monkeypatch.setattr(build, "LIB_PATH", str(lib))
    monkeypatch.setattr(build, "HOST_PATH", str(host))
    monkeypatch.setattr(build, "hipcc_path", lambda: "hipcc")

    def run(fail, text):
        def step(cmd, verbose):
            out = cmd[cmd.index("-o") + 1]
            with open(out, "w") as f:
                f.write(text)
            if fail and fail in out:
                raise RuntimeError("no compiler")
        return step
    monkeypatch.setattr(build, "_run", run(None, "old"))
    assert build.build(False) == str(lib)
    monkeypatch.setattr(build, "_run", run(broken, "new"))
    with pytest.raises(RuntimeError):
        build.build(False)
    assert lib.read_text() == host.read_text() == "old" and len(list(tmp_path.iterdir())) == 2
    monkeypatch.setattr(build, "_run", run(None, "new"))
    build.build(False)
    assert lib.read_text() == host.read_text() == "new" and len(list(tmp_path.iterdir())) == 2
