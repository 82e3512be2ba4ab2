"""The compiled host path is an addition: without its module, with one of another torch or with a library that lacks an entry point of it, the public functions
say so once and serve calls by their own statements.  And it is there: ordinary tensors are not served by those statements without being noticed."""
import os
import subprocess
import sys
import warnings

import pytest
import torch

import gcnasm_amd as g
from gcnasm_amd import api

FAST = ("_fast_gemm", "_fast_quantize", "_fast_quantize_mxfp4", "_fast_encode", "_fast_decode")
CSRC = os.path.join(os.path.dirname(os.path.abspath(g.__file__)), "csrc")


class OldLibrary:
    def __init__(self, library):
        self.library = library

    def __getattr__(self, name):
        if name == "a8w8_quantize_ws":
            raise AttributeError(name)
        return getattr(self.library, name)


def _no_module(monkeypatch):
    monkeypatch.delattr(g, "_binding", raising=False)
    monkeypatch.setitem(sys.modules, "gcnasm_amd._binding", None)


def _module_of_another_torch(monkeypatch):
    from gcnasm_amd import _binding
    monkeypatch.setattr(_binding, "torch_build", "1.0 f00")


def _older_library(monkeypatch):
    monkeypatch.setattr(api, "_lib", OldLibrary(api.lib()))


@pytest.fixture(params=[_no_module, _module_of_another_torch, _older_library], ids=lambda f: f.__name__)
def without_the_module(request, monkeypatch):
    for name in FAST:
        monkeypatch.setattr(api, name, getattr(api, name))      # (put back afterwards)
    request.param(monkeypatch)
    with pytest.warns(RuntimeWarning, match="_binding.so is not used"):
        api._connect()


def test_statements_take_over(without_the_module):
    x = torch.zeros(4, 128)
    with warnings.catch_warnings():
        warnings.simplefilter("error")      # once is enough
        assert api._fast_quantize(x, g.ROWCOL, 1) is None and api._fast_gemm(0) is None and api._fast_encode(x, 0, 0) is None
        with pytest.raises(ValueError, match="GPU"):
            g.quantize(x, g.ROWCOL)


@pytest.mark.gpu
def test_same_results_without_the_module(without_the_module):
    x, w = torch.randn(48, 512, device="cuda"), torch.randn(256, 512, device="cuda")
    for mode in (g.TENSOR, g.ROWCOL):
        (a, sa), (b, sb) = g.quantize(x, mode), g.quantize(w, mode)
        c = g.gemm(a, b, sa, sb, mode, c_dtype=g.FP32)
        assert (c - x @ w.T).norm() < 0.1 * c.norm()
    assert torch.equal(g.cvt_e4m3_to_f32(g.cvt_f32_to_e4m3(x)).sign(), g.cvt_f32_to_e4m3(x).view(torch.float8_e4m3fn).float().sign())


def test_library_alone():
    """`make lib` asks for neither Python nor torch."""
    plan = subprocess.run(["make", "-n", "-B", "-C", CSRC, "lib", "PY=/nonexistent"], capture_output=True, text=True)
    assert plan.returncode == 0 and "libmi355a8w8" in plan.stdout and "binding.cpp" not in plan.stdout and "nonexistent" not in plan.stdout + plan.stderr
    whole = subprocess.run(["make", "-n", "-B", "-C", CSRC], capture_output=True, text=True)
    assert whole.returncode == 0 and "binding.cpp" in whole.stdout and "-DA8W8_TORCH_BUILD='\"" + api._torch_build() in whole.stdout
    none = subprocess.run(["make", "-n", "-B", "-C", CSRC, "PY=/nonexistent"], capture_output=True, text=True)
    assert none.returncode == 0 and "binding.cpp" not in none.stdout and "no torch" in none.stdout
