"""Where the native host calls cannot be used (csrc/host_calls.cpp: not built, or for another torch or
Python) every call goes the general way behind them, with one warning."""
import sys
import types
import warnings

import pytest
import torch

import tritonops_amd
from tritonops_amd import _lib


@pytest.fixture
def unloaded(monkeypatch):
    monkeypatch.setattr(_lib, "_native", None)
    monkeypatch.delattr(tritonops_amd, "_native", raising=False)


def _answers(module):
    return [getattr(module, name)(1, 2) for name in ("rms_fwd", "rms_bwd", "dense_fwd", "dense_bwd", "sparse_fwd", "decode")]


@pytest.mark.parametrize("module", [None, types.SimpleNamespace(built_for=("1.0", "3.10")), types.SimpleNamespace()],
                         ids=["missing", "other_torch", "no_versions"])
def test_the_general_way_without_it(monkeypatch, unloaded, module):
    monkeypatch.setitem(sys.modules, "tritonops_amd._native", module)
    with pytest.warns(RuntimeWarning, match="_native.so"):
        got = _lib.native()
    assert _answers(got) == [None] * 6
    with warnings.catch_warnings():
        warnings.simplefilter("error")
        assert _lib.native() is got


def test_as_built_it_is_used(unloaded):
    with warnings.catch_warnings():
        warnings.simplefilter("error")
        module = _lib.native()
    assert module.built_for == (torch.__version__, "%d.%d" % sys.version_info[:2])
    assert all(hasattr(module, name) for name in ("rms_fwd", "rms_bwd", "dense_fwd", "dense_bwd", "sparse_fwd", "decode"))
