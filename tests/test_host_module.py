"""Loading the native host module (csrc/host.cpp): the library works without
it, and a module compiled against another C ABI is not used."""
import ctypes
import shutil

import pytest

from mxfp8gg import _lib


@pytest.fixture
def fresh(monkeypatch):
    """_lib as before its first load."""
    if not _lib.LIB_PATH.exists():
        pytest.skip("libmxgg.so is not built")
    monkeypatch.setattr(_lib, "_lib", None)
    monkeypatch.setattr(_lib, "_native", None)
    return monkeypatch


@pytest.mark.parametrize("how", ["missing", "unreadable"])
def test_library_loads_without_the_host_module(fresh, tmp_path, how):
    path = tmp_path / _lib.HOST_PATH.name
    if how == "unreadable":
        path.write_bytes(b"no shared object")
    fresh.setattr(_lib, "HOST_PATH", path)
    with pytest.warns(RuntimeWarning, match="native host module"):
        lib = _lib.load()
    assert lib.mxgg_abi_version() == _lib.ABI_VERSION
    assert _lib.native() is None        # every op then takes its Python form


def test_a_module_of_another_abi_is_refused(fresh, tmp_path):
    """bind() against a library that reports another version raises and leaves
    the module as it was."""
    if not _lib.HOST_PATH.exists():
        pytest.skip("the host module is not built")
    other = ctypes.CFUNCTYPE(ctypes.c_int)(lambda: _lib.ABI_VERSION + 1)
    path = tmp_path / _lib.HOST_PATH.name
    shutil.copy(_lib.HOST_PATH, path)   # a module of its own: the loaded one stays bound
    fresh.setattr(_lib, "HOST_PATH", path)
    lib = _lib.load()
    address = {n: ctypes.cast(getattr(lib, n), ctypes.c_void_p).value for n in _lib.SIGNATURES}
    address["mxgg_abi_version"] = ctypes.cast(other, ctypes.c_void_p).value
    with pytest.raises(RuntimeError, match="ABI version"):
        _lib.native().bind(address)


def test_both_load_together(fresh):
    if not _lib.HOST_PATH.exists():
        pytest.skip("the host module is not built")
    _lib.load()
    assert _lib.native() is not None
