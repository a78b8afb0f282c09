"""The native call module is loaded for the interpreter and torch that it was built for, and for no others."""

from __future__ import annotations

import sys

import torch

from attnarc_amd import _native
from attnarc_amd import build as hip_build


def test_built_module_is_used(monkeypatch):
    monkeypatch.setattr(_native, "_calls", None)
    assert _native.calls().__name__ == "_loom_hip_calls"


def test_other_versions_have_other_files(monkeypatch):
    built = hip_build.calls_path()
    assert sys.implementation.cache_tag in built and torch.__version__ in built
    monkeypatch.setattr(torch, "__version__", torch.__version__ + ".other")
    assert hip_build.calls_path() != built


def test_calls_go_through_python_without_one(monkeypatch):
    monkeypatch.setattr(_native, "_calls", None)
    monkeypatch.setattr(torch, "__version__", torch.__version__ + ".other")  # nothing was built for it
    calls = _native.calls()
    assert getattr(calls, "__name__", "") != "_loom_hip_calls"
    assert calls.decode_extended(*range(15)) is None
    assert calls.decode_views(*range(8)) is None and calls.rope_write(*range(10)) is None
    assert _native.calls() is calls
