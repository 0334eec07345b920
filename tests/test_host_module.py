"""The native host module (csrc/host.cpp) is a fast path only: without it every
call keeps the Python path to the libraries (runs without a GPU)."""

from __future__ import annotations

import ctypes
import sys
import types
import warnings

import pytest

import flashinfer_competition_codebase_amd as gdn
from flashinfer_competition_codebase_amd import _lib

MODULE = "flashinfer_competition_codebase_amd._gdn_host"


@pytest.fixture
def unbound(monkeypatch):
    monkeypatch.setattr(_lib, "bound_host", None)
    monkeypatch.setattr(_lib, "_host_error", None, raising=False)
    monkeypatch.setattr(_lib, "_host_halves", set(), raising=False)
    monkeypatch.delattr(gdn, "_gdn_host", raising=False)


@pytest.mark.parametrize("module", [None, types.SimpleNamespace(torch_version="1.0.0")])
def test_a_module_that_does_not_load_is_no_error(module, unbound, monkeypatch):
    """None: the import fails; else compiled against another torch."""
    if module is not None:
        monkeypatch.setattr(gdn, "_gdn_host", module, raising=False)
    monkeypatch.setitem(sys.modules, MODULE, module)
    with pytest.warns(RuntimeWarning, match="native host module"):
        _lib.bind_host()
    assert _lib.bound_host is None
    with warnings.catch_warnings():
        warnings.simplefilter("error")
        _lib.bind_host()                            # said once
    assert _lib.bound_host is None


@pytest.mark.parametrize("half,other", [("decode", "get_prefill_lib"), ("prefill", "get_lib")])
def test_each_half_needs_its_own_library_only(half, other, unbound, monkeypatch):
    def missing():
        raise RuntimeError("library not found")
    monkeypatch.setattr(_lib, other, missing)
    _lib.bind_host(**{{"decode": "prefill", "prefill": "decode"}[half]: False})
    assert _lib.bound_host is not None and _lib._host_halves == {half}


def test_a_bound_module_is_bound_once(unbound, monkeypatch):
    _lib.bind_host()
    assert _lib._host_halves == {"decode", "prefill"}
    host = _lib.bound_host
    monkeypatch.setattr(ctypes, "cast", None)       # nothing left to bind
    _lib.bind_host()
    assert _lib.bound_host is host
