"""The choice between the native host path and the general way, without a GPU."""
import os
import subprocess
import sys
import sysconfig
import warnings
from importlib import import_module

import pytest
import torch


def test_general_way_where_the_module_does_not_load(pkg, monkeypatch):
    """No native module: one warning, and every call declines instead of raising."""
    lib = import_module("fni8serve_amd._lib")
    monkeypatch.setitem(sys.modules, "fni8serve_amd._host", None)
    monkeypatch.delattr(pkg, "_host", raising=False)
    monkeypatch.setattr(lib, "_host", None)
    with warnings.catch_warnings(record=True) as seen:
        warnings.simplefilter("always")
        for name in ("linear", "gemm", "mlp", "rmsnorm", "moe"):
            assert getattr(lib.host(), name)(None, 1) is None
    assert [w.category for w in seen] == [RuntimeWarning]


def test_module_of_another_build_is_not_used(pkg, monkeypatch):
    """The module is tied to one Python (its file name) and one torch (checked)."""
    lib = import_module("fni8serve_amd._lib")
    native = import_module("fni8serve_amd._host")
    assert native.__file__.endswith("_host" + sysconfig.get_config_var("EXT_SUFFIX"))
    monkeypatch.setattr(lib, "_host", None)
    assert lib.host() is native
    monkeypatch.setattr(lib, "_host", None)
    monkeypatch.setattr(torch, "__version__", "0.0.0")
    with pytest.warns(RuntimeWarning, match="0.0.0"):
        assert lib.host().linear(None) is None


@pytest.mark.parametrize("python,host", [(sys.executable, True), (sys.executable + " -S", False)])
def test_make_without_torch_builds_the_library(pkg, python, host):
    """`make` in csrc (here its plan): without torch (-S: no site-packages) the C library
    is the whole build, with it the extension module too."""
    csrc = os.path.join(os.path.dirname(pkg.__file__), "csrc")
    plan = subprocess.run(["make", "-n", "-B", "-C", csrc, f"PYTHON={python}"],
                          capture_output=True, text=True, timeout=60)
    assert plan.returncode == 0 and plan.stderr == ""
    assert "-shared -o ../libfni8amd.so" in plan.stdout
    assert ("host.cpp" in plan.stdout) == host


_SURGERY = {
    "hook": lambda m, mp: m.register_forward_hook(lambda *a: None),
    "pre_hook": lambda m, mp: m.register_forward_pre_hook(lambda *a: None),
    "own_forward": lambda m, mp: mp.setattr(m, "forward", lambda x: x, raising=False),
    "class_forward": lambda m, mp: mp.setattr(type(m), "forward", lambda self, x: x),
    "class_call": lambda m, mp: mp.setattr(type(m), "__call__", lambda self, x: x, raising=False),
    "compiled": lambda m, mp: mp.setattr(m, "_compiled_call_impl", lambda x: x),
    "subclass": lambda m, mp: setattr(m, "__class__", type("Sub", (type(m),), {})),
    "own_rule": lambda m, mp: mp.setattr(m, "_int8_ok", lambda x: False, raising=False),
    "class_rule": lambda m, mp: mp.setattr(type(m), "_int8_ok", lambda self, x: False, raising=False),
}


@pytest.mark.parametrize("surgery", sorted(_SURGERY))
@pytest.mark.parametrize("part", ["gate_up_proj", "down_proj", "act_fn"])
def test_bare_sees_module_surgery(pkg, monkeypatch, surgery, part):
    """The one-call MLP is for untouched parts: whatever else a call would run shows."""
    bare = import_module("fni8serve_amd.layers.mlp").bare
    qt = [pkg.QTensor(torch.zeros(n, k, dtype=torch.int8), torch.ones(n), scheme="per_row_i8")
          for n, k in ((16, 8), (8, 8))]
    m = getattr(pkg.GatedMLP(*qt), part)
    cls = type(m)
    assert bare(m, cls)
    _SURGERY[surgery](m, monkeypatch)
    if part == "act_fn" and surgery.endswith("rule"):
        return  # an activation has no such rule
    assert not bare(m, cls)


@pytest.mark.parametrize("owner", ["instance", "class"])
@pytest.mark.parametrize("step", ["route", "experts_grouped", "experts_grouped_w4"])
def test_moe_steps_replaced(pkg, monkeypatch, owner, step):
    """SparseMoE's one call is for the steps that the class was defined with."""
    ops = import_module("fni8serve_amd.ops")
    monkeypatch.setattr(ops, "sparse_moe", lambda *a: "one call")
    qt = [pkg.QTensor(torch.zeros(n, k, dtype=torch.int8), torch.ones(n), scheme="per_row_i8")
          for n, k in ((16, 8), (8, 8))]
    moe = pkg.SparseMoE(gate=torch.zeros(2, 8), experts=[qt, qt], top_k=1)
    x = torch.zeros(3, 8)
    assert moe._native(x) == "one call"
    monkeypatch.setattr(moe if owner == "instance" else pkg.SparseMoE, step, lambda *a: None,
                        raising=False)
    assert moe._native(x) is None
