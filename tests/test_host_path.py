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
