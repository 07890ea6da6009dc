"""kvq._torch_calls belongs to one library, one torch and one Python: the package binds it only where all three are
the ones it was compiled for, and a failed build leaves no older file behind. No GPU."""
import importlib.util
import os
import sys
import types
import warnings

import pytest
import torch

import kvq
from kvq import _native
from kvq import cuda_kernels as ck

REPO = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def _load_calls():
    with warnings.catch_warnings(record=True) as w:
        warnings.simplefilter("always")
        return _native.torch_calls(), [str(x.message) for x in w]


def test_the_built_module_is_bound():
    calls, warned = _load_calls()
    assert calls is not None and not warned
    assert calls.BUILT_FOR == _native.calls_built_for()


@pytest.mark.parametrize("other", ["abi", "torch", "python"])
def test_a_module_built_for_something_else_is_not_bound(other, monkeypatch):
    """The operators then run the Python path; one warning names what the module was built for."""
    _native.load()
    if other == "abi":
        monkeypatch.setattr(_native, "ABI_VERSION", _native.ABI_VERSION + 1)
    elif other == "torch":
        monkeypatch.setattr(torch, "__version__", torch.__version__ + ".other")
    else:
        monkeypatch.setattr(sys, "version_info", (sys.version_info[0], sys.version_info[1] + 1, 0, "final", 0))
    monkeypatch.setattr(ck, "_EXT", None)
    with warnings.catch_warnings(record=True) as w:
        warnings.simplefilter("always")
        e = ck.ext()
    assert e.calls is None
    assert len(w) == 1 and "_torch_calls" in str(w[0].message)
    assert not ck._served(e, "quant_cache", *[None] * 8)


def test_a_module_without_the_record_is_not_bound(monkeypatch):
    """A file left from before the record existed: never called, not even to bind it."""
    monkeypatch.setitem(sys.modules, "kvq._torch_calls", old := types.ModuleType("kvq._torch_calls"))
    monkeypatch.setattr(kvq, "_torch_calls", old, raising=False)
    calls, warned = _load_calls()
    assert calls is None and len(warned) == 1


def _build_module(tmp_path, monkeypatch, hipcc, cxx):
    spec = importlib.util.spec_from_file_location("kvq_build", os.path.join(REPO, "int8-kvcache_amd", "build.py"))
    b = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(b)
    for name, ok in (("HIPCC", hipcc), ("CXX", cxx)):
        tool = tmp_path / name
        tool.write_text('#!/bin/sh\nwhile [ "$1" != -o ]; do shift; done\necho new > "$2"\n' + ("" if ok else "echo no; exit 1\n"))
        tool.chmod(0o755)
        monkeypatch.setattr(b, name, str(tool))
    for name in ("OUT", "CALLS_OUT"):
        monkeypatch.setattr(b, name, str(tmp_path / (name + ".so")))
        (tmp_path / (name + ".so")).write_text("old")
    return b


@pytest.mark.parametrize("hipcc,cxx", [(True, True), (True, False), (False, True), (False, False)])
def test_a_failed_build_leaves_no_older_file(hipcc, cxx, tmp_path, monkeypatch):
    b = _build_module(tmp_path, monkeypatch, hipcc, cxx)
    if hipcc and cxx:
        b.build()
    else:
        with pytest.raises(RuntimeError, match="failed"):
            b.build()
    for name, ok in (("OUT", hipcc), ("CALLS_OUT", cxx)):
        path = tmp_path / (name + ".so")
        assert path.exists() == ok and (not ok or path.read_text() == "new\n")
    assert not list(tmp_path.glob("*.tmp"))
