"""The choice between the native host path and the general way, without a GPU."""
import sys
import warnings
from importlib import import_module


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
