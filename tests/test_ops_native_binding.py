"""When ops uses the separately compiled _ops_native.so (CPU only): built for the running torch and Python and with
the header that the library was built with, and in no other case, however well it loads."""
from __future__ import annotations

import sys
from types import SimpleNamespace

import pytest

torch = pytest.importorskip("torch")

from v7multiplikator_amd import _lib, build, ops  # noqa: E402


def bound(L=None):
    return not isinstance(ops._bind_native(L or _lib.load()), ops._NoNative)


def test_the_built_module_is_bound():
    assert bound()
    assert f'-DV7G_HEADER_TAG="{_lib.load().v7g_header_tag().decode()}"' == build.header_tag_flag()


def test_another_header_is_refused():
    L = _lib.load()
    entries = {n: getattr(L, n) for n in _lib.SIGNATURES}
    assert bound(SimpleNamespace(**entries))
    assert not bound(SimpleNamespace(**{**entries, "v7g_header_tag": lambda: b"0123456789abcdef"}))


def test_another_torch_is_refused(monkeypatch):
    with monkeypatch.context() as m:
        m.setattr(torch.version, "git_version", "0" * 40)
        assert not bound()
    with monkeypatch.context() as m:
        m.setattr(torch, "__version__", "2.10.1")
        assert not bound()
    assert bound()


def test_another_python_is_refused(monkeypatch):
    monkeypatch.setattr(sys, "version_info", (3, sys.version_info[1] + 1))
    assert not bound()


def test_a_module_without_the_attributes_is_refused(monkeypatch, tmp_path):
    (tmp_path / "_ops_native.py").write_text("def bind(*args): raise AssertionError('bound')\n")
    monkeypatch.setattr(ops, "_NATIVE_PATH", str(tmp_path / "_ops_native.py"))
    assert not bound()
