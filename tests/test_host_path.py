"""The choice between the native host path and the general way, without a GPU."""
import os
import subprocess
import sys
import warnings
from importlib import import_module

import pytest


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
