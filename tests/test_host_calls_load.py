"""The native host calls are an accelerator of libtu_hip.so's Python route, not a
condition of it: a module that is missing, does not load or was built against
another torch leaves the general route, with one warning."""
from __future__ import annotations

import sys
import types
import warnings

import pytest
import torch

import comfyui_turing_utils_kernel as package
from comfyui_turing_utils_kernel import _lib

NAME = "comfyui_turing_utils_kernel._host_calls"
CALLS = ("int8_linear", "sageattn", "w8a8attn")


@pytest.fixture
def module(monkeypatch):
    """Makes `from . import _host_calls` find the given entry of sys.modules."""
    def put(entry):
        monkeypatch.setattr(_lib, "_host", None)
        monkeypatch.delattr(package, "_host_calls", raising=False)
        monkeypatch.setitem(sys.modules, NAME, entry)
    return put


def _other_torch():
    m = types.ModuleType(NAME)
    m.torch_version = "0.0.0"
    return m


@pytest.mark.parametrize("entry,reason", [
    (lambda: None, "cannot be loaded"),                           # missing, or a symbol that does not resolve
    (_other_torch, "was built against torch 0.0.0"),
    (lambda: types.ModuleType(NAME), "was built against torch None"),
])
def test_unusable_module_means_the_general_route(module, entry, reason):
    module(entry())
    with pytest.warns(RuntimeWarning, match=reason):
        calls = _lib.host_calls()
    assert all(getattr(calls, name)(1, 2, 3) is None for name in CALLS)
    with warnings.catch_warnings():
        warnings.simplefilter("error")
        assert _lib.host_calls() is calls  # said once


def test_built_module_is_used():
    calls = _lib.host_calls()
    assert calls.torch_version == torch.__version__
    assert all(callable(getattr(calls, name)) for name in CALLS)


def test_stream_handle_without_the_private_accessor():
    assert callable(_lib.raw_stream) and callable(_lib._stream_handle)
