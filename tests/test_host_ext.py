"""The extension with the native host calls can be done without: where it does
not load, the calls take the Python path to the same kernels."""
import sys
import types

import pytest
import torch


@pytest.fixture()
def fresh(monkeypatch):
    """host() as before its first call, with `module` (None: cannot be
    imported) in the extension's place."""
    import flashvsr_sm89_ops
    from flashvsr_sm89_ops import _lib

    def put(module):
        monkeypatch.setattr(_lib, "_host", None)
        monkeypatch.setitem(sys.modules, "flashvsr_sm89_ops._fvsr_host", module)
        monkeypatch.delattr(flashvsr_sm89_ops, "_fvsr_host", raising=False)
        if module is not None:
            monkeypatch.setattr(flashvsr_sm89_ops, "_fvsr_host", module, raising=False)
        return _lib
    return put


def _stand_in(version):
    m = types.ModuleType("flashvsr_sm89_ops._fvsr_host")
    if version is not None:
        m.torch_version = version
    m.bound = []
    m.bind = lambda *a: m.bound.append(a)
    m.quantize = m.gemm = lambda *a: "native"
    return m


def test_missing_extension_leaves_calls_to_the_python_path(fresh):
    _lib = fresh(None)
    with pytest.warns(RuntimeWarning, match="native host calls are off"):
        h = _lib.host()
    assert h.quantize(1, 2, 3) is None and h.gemm(1, 2, 3, 4, 5, 6) is None
    assert _lib.host() is h  # once


@pytest.mark.parametrize("version", ["1.0.0", None])
def test_extension_of_another_torch_is_not_used(fresh, version):
    m = _stand_in(version)
    _lib = fresh(m)
    with pytest.warns(RuntimeWarning, match=f"built with torch {version or 'of another version'}"):
        h = _lib.host()
    assert h.gemm() is None and not m.bound


def test_extension_of_this_torch_is_bound(fresh):
    m = _stand_in(torch.__version__)
    _lib = fresh(m)
    h = _lib.host()
    assert h is m and len(m.bound) == 1 and all(m.bound[0]) and len(m.bound[0]) == 4


def test_built_extension_names_its_torch():
    from flashvsr_sm89_ops import _fvsr_host
    assert _fvsr_host.torch_version == torch.__version__
