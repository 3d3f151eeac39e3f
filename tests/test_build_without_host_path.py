"""The native host path (``_host.so``) is an extra: the kernel library builds without it, a machine that cannot build or load
it gets a message, and the operators then run the Python form of the same host logic."""
import os
import shutil
import subprocess
import sys
import warnings

import pytest
import torch

import __graft_entry__
import flag_attn
import flagattention_amd
from flagattention_amd import _lib

CSRC = os.path.join(os.path.dirname(os.path.abspath(flagattention_amd.__file__)), "csrc")


def test_kernel_library_is_built_without_python():
    out = subprocess.run(["make", "-n", "-B", "-C", CSRC, "PYTHON=/nonexistent/python"], capture_output=True, text=True, check=True)
    assert "libflagattn_hip.so" in out.stdout and "host.cpp" not in out.stdout and "torch" not in out.stdout
    assert "nonexistent" not in out.stderr


def test_build_goes_on_where_the_host_path_cannot_be_built(tmp_path, monkeypatch, capfd):
    for d in ("package/csrc", "include"):
        os.makedirs(tmp_path / d)
    for name in ("Makefile", "host.cpp"):
        shutil.copy(os.path.join(CSRC, name), tmp_path / "package" / "csrc")
    (tmp_path / "include" / "flagattn.h").touch()
    (tmp_path / "package" / "libflagattn_hip.so").touch()
    monkeypatch.setattr(__graft_entry__, "CSRC", str(tmp_path / "package" / "csrc"))
    assert not __graft_entry__.build_host(python="/bin/false")      # an interpreter that knows no torch
    assert "_host.so was not built" in capfd.readouterr().err


@pytest.fixture
def no_host(monkeypatch):
    monkeypatch.setattr(_lib, "_native", None)
    monkeypatch.setitem(sys.modules, "flagattention_amd._host", None)    # importing it raises ImportError
    monkeypatch.delattr(flagattention_amd, "_host", raising=False)


def test_missing_host_path_is_reported_once(no_host):
    with pytest.warns(RuntimeWarning, match="make -C flagattention_amd/csrc host"):
        native = _lib.native()
    with warnings.catch_warnings():
        warnings.simplefilter("error")
        assert _lib.native() is native
    assert native.flash() is native.piecewise() is native.paged() is NotImplemented


@pytest.mark.gpu
@pytest.mark.filterwarnings("ignore:the native host path is not used")
def test_operators_without_the_host_path(no_host):
    gen = torch.Generator(device="cuda").manual_seed(2)
    q, k, v, q2, k2 = (torch.randn(1, 4, 200, 64, device="cuda", dtype=torch.float16, generator=gen).requires_grad_() for _ in range(5))
    lens, table = torch.tensor([40, 9], dtype=torch.int32, device="cuda"), torch.arange(6, device="cuda").reshape(2, 3)
    cache = torch.randn(6, 4, 16, 64, device="cuda", dtype=torch.float16, generator=gen)
    query = q.detach()[0, :, :2].transpose(0, 1).contiguous()

    def results():
        o, p = flag_attn.flash_attention(q, k, v, True), flag_attn.piecewise_attention(q, k, q2, k2, v, 50, True)
        return (o, p, flag_attn.paged_attention(query, cache, cache, lens, table, 0.125, 40)) + \
            torch.autograd.grad(o, (q, k, v), q.detach()) + torch.autograd.grad(p, (q, k, q2, k2, v), q.detach())

    python = results()
    assert _lib.native() is _lib.PythonForm
    _lib._native = None
    sys.modules.pop("flagattention_amd._host")
    for a, b in zip(python, results()):
        assert torch.equal(a, b)
