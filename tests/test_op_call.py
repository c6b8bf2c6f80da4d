"""Op.run's native call against the ctypes one: the same status and error for every kind of argument. No GPU: the library checks
its operands before it launches anything."""
import ctypes as C
import enum
import importlib.machinery
import importlib.util
import os
import sys
import sysconfig
import warnings

import pytest

import tvx_case as TC


class _Tensor:
    def __init__(self, address):
        self.address = address

    def data_ptr(self):
        return self.address


def _needs_binding(T):
    if not os.path.exists(os.path.join(sysconfig.get_paths()["include"], "Python.h")):
        pytest.skip("no headers of Python: the call goes through ctypes")
    assert T._run is not T._ctypes_run, "the native call is not built"


@pytest.mark.parametrize("native", [False, True], ids=["ctypes", "native"])
def test_run_arguments(monkeypatch, native):
    T = TC.tvx()
    T.lib()
    if native:
        _needs_binding(T)
    else:
        monkeypatch.setattr(T, "_run", T._ctypes_run)
    t = _Tensor(4096)
    for handle in (None, C.c_void_p(None)):
        for stream in (None, 0, C.c_void_p(0), C.POINTER(C.c_int)()):
            op = T.Op(handle)
            with pytest.raises(T.TvxError, match="null operator") as err:
                op.run(t, None, 4096, stream)
            assert err.value.status == T.E_INVALID
    with pytest.raises(AttributeError):
        T.Op(None).run(t, "text", t)


def test_native_call_passes_addresses():
    T = TC.tvx()
    L = T.lib()
    _needs_binding(T)
    seen = []
    run = C.CFUNCTYPE(C.c_int, *[C.c_void_p] * 5)(lambda *a: seen.append(a) or -3)
    module = T._run.__self__
    module.bind(C.cast(run, C.c_void_p).value, C.c_void_p)
    try:
        high = (1 << 47) + 16
        assert T._run(C.c_void_p(high), _Tensor(high + 1), None, high + 2, C.c_void_p(7)) == -3
        assert T._run(5, 6, _Tensor(0), _Tensor(8), None) == -3
    finally:
        module.bind(C.cast(L.tvx_op_run, C.c_void_p).value, C.c_void_p)
    assert seen == [((1 << 47) + 16, (1 << 47) + 17, None, (1 << 47) + 18, 7), (5, 6, None, 8, None)]


@pytest.mark.parametrize("native", [False, True], ids=["ctypes", "native"])
def test_no_truth_of_not_implemented(monkeypatch, native):
    """A pointer type that only ctypes knows gives NotImplemented, whose truth warns and in later versions raises."""
    T = TC.tvx()
    T.lib()
    if not native:
        monkeypatch.setattr(T, "_run", T._ctypes_run)
    with warnings.catch_warnings():
        warnings.simplefilter("error")
        with pytest.raises(T.TvxError, match="null operator"):
            T.Op(None).run(_Tensor(4096), None, 4096, C.POINTER(C.c_int)())


def test_run_loads_the_library(monkeypatch):
    T = TC.tvx()
    spec = importlib.util.spec_from_file_location("tvx_unloaded", T.__file__, submodule_search_locations=T.__path__)
    unloaded = importlib.util.module_from_spec(spec)
    monkeypatch.setitem(sys.modules, "tvx_unloaded", unloaded)
    spec.loader.exec_module(unloaded)
    with pytest.raises(unloaded.TvxError, match="null operator"):
        unloaded.Op(None).run(4096, None, 4096)


class _Code(enum.Enum):
    OTHER = 4096


@pytest.mark.parametrize("native", [False, True], ids=["ctypes", "native"])
def test_what_is_no_pointer_is_refused(monkeypatch, native):
    T = TC.tvx()
    T.lib()
    if not native:
        monkeypatch.setattr(T, "_run", T._ctypes_run)
    for wrong in (C.c_int(4096), C.c_uint64(4096), _Code.OTHER):
        with pytest.raises(C.ArgumentError):
            T.Op(None).run(4096, None, 4096, wrong)
        with pytest.raises(C.ArgumentError):
            T.Op(wrong).run(4096, None, 4096)


@pytest.mark.parametrize("native", [False, True], ids=["ctypes", "native"])
def test_addresses_of_every_kind(monkeypatch, native):
    T = TC.tvx()
    T.lib()
    if not native:
        monkeypatch.setattr(T, "_run", T._ctypes_run)
    for address in (None, 4096, C.c_void_p(4096), C.POINTER(C.c_int)()):
        with pytest.raises(T.TvxError, match="null operator"):
            T.Op(None).run(_Tensor(address), None, _Tensor(4096))
    with pytest.raises(C.ArgumentError):
        T.Op(None).run(_Tensor(1.5), None, _Tensor(4096))


def test_a_binding_that_does_not_load_leaves_the_call_to_ctypes(monkeypatch, tmp_path):
    """A file of another interpreter's ABI, or a broken one."""
    T = TC.tvx()
    L = T.lib()
    (tmp_path / "lib").mkdir()
    (tmp_path / "lib" / ("tvx_call" + importlib.machinery.EXTENSION_SUFFIXES[0])).write_bytes(b"no library")
    (tmp_path / "lib" / "tvx_call.so").write_bytes(b"no library")
    monkeypatch.setattr(T, "PKG_DIR", str(tmp_path))
    assert T._native_run(L) is T._ctypes_run


def test_a_build_without_headers_leaves_no_binding_behind(monkeypatch, tmp_path):
    build = importlib.import_module("tim-vx_amd.build")
    (tmp_path / "lib").mkdir()
    for name in ("tvx_call" + importlib.machinery.EXTENSION_SUFFIXES[0], "tvx_call.so"):
        (tmp_path / "lib" / name).write_bytes(b"")
    monkeypatch.setattr(build, "PKG_DIR", str(tmp_path))
    monkeypatch.setattr(sysconfig, "get_paths", lambda: {"include": str(tmp_path)})
    build.build_binding()
    assert os.listdir(str(tmp_path / "lib")) == []
