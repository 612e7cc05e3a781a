"""The extension module that calls libfa_gpu.so (csrc/host/fa_call.cpp) against
ctypes on the same library: refusals the library makes before any HIP call, so no
GPU is needed."""

from __future__ import annotations

import ctypes
import sysconfig

import pytest

from frame_analytics_amd import _build, _cabi

if not _build.library_path().exists():  # pragma: no cover
    pytest.skip("libfa_gpu.so is not built", allow_module_level=True)


@pytest.fixture(scope="module")
def both():
    lib, _ = _cabi.load_gpu()
    callers = _cabi.load_callers(lib)
    assert callers, "the extension module did not load"
    return lib, callers


def _null_args(name):
    """One refused call: null pointers, zero sizes."""
    kinds, _ = _cabi.SIGNATURES[name]
    return [None if k is ctypes.c_void_p else 0.5 if k is ctypes.c_double else 0 for k in kinds]


def test_statuses_match_ctypes(both):
    lib, callers = both
    for name, fast in callers.items():
        args = _null_args(name)
        want = getattr(lib, name)(*args)
        assert want != 0 and fast(*args) == want, name


def test_arguments_reach_their_places(both):
    """Each of these refusals depends on one argument after doubles, arrays and
    addresses: a shifted or narrowed argument gives another status."""
    lib, callers = both
    fast = callers["fa_gpu_ssim_once"]
    buf = ctypes.create_string_buffer(4096)
    p = ctypes.addressof(buf)
    strides = (ctypes.c_int64 * 3)(3 * 64 * 64, 64 * 64, 32)  # rows of 64 overlap
    luma = (ctypes.c_double * 4)(0.3, 0.6, 0.1, 0.0)

    def args(xs=None, lw=None, k=11, bpp=None, c=1):
        n = ctypes.c_int(0)
        assert lib.fa_gpu_ssim_workspace(64, 64, 11, ctypes.byref(n)) == 0
        return (p, p, 0, 1, c, 64, 64, xs, None, lw, p, k, 127.5, 6.5, 58.5, None, p,
                n.value if bpp is None else bpp, None, p, p, 0, None)

    for kw in ({"xs": strides}, {"lw": luma}, {"k": 4}, {"bpp": 1}, {"c": 0}, {"c": -1}):
        want = lib.fa_gpu_ssim_once(*args(**kw))
        assert want > 0 and fast(*args(**kw)) == want, kw


def test_wrong_arguments_raise(both):
    _, callers = both
    fast = callers["fa_gpu_gmsd_backward"]
    args = _null_args("fa_gpu_gmsd_backward")
    with pytest.raises(TypeError):
        fast(*args[:-1])
    with pytest.raises(TypeError):
        fast(*args, None)
    with pytest.raises(TypeError):
        fast("x", *args[1:])
    with pytest.raises(TypeError):
        fast(*args[:7], "x", *args[8:])


def test_build_without_python_headers(monkeypatch, tmp_path, capsys):
    """A machine that cannot compile the module still gets the libraries, the
    fallback to ctypes, and no build that stays stale for the module's sake."""
    monkeypatch.setattr(_build, "LIBDIR", tmp_path)
    monkeypatch.setattr(_build, "python_include", lambda: tmp_path / "none")
    made = []
    real = _build._run

    def run(cmd, verbose):  # the kernels' compiler leaves its outputs, nothing else
        if cmd[0] == "hipcc-stub":
            made.append(cmd[-1])
            open(cmd[-1], "wb").close()
        else:
            real(cmd, verbose)

    monkeypatch.setattr(_build, "_run", run)
    monkeypatch.setattr(_build, "hipcc", lambda: "hipcc-stub")
    monkeypatch.setattr(_build, "PKG", tmp_path)
    _build.call_module_path().write_bytes(b"of an earlier build")
    assert _build.build() == _build.library_path() and _build.library_path().exists()
    assert len(made) == len(_build.sources()) + 2
    assert not _build.call_module_path().exists()
    assert "Python.h" in capsys.readouterr().err
    assert not _build.is_stale()
    assert _cabi.load_callers(None) == {}


def test_module_of_another_interface_is_not_called(both, monkeypatch, tmp_path):
    """A module whose prototypes, ABI version or interpreter are not those of the
    library and of ctypes: its entries are left to ctypes."""
    lib, callers = both
    name = "fa_gpu_gmsd_once"
    args, res = _cabi.SIGNATURES[name]
    swapped = list(args)  # the same count: a double for an int
    swapped[swapped.index(ctypes.c_int)] = ctypes.c_double
    monkeypatch.setitem(_cabi.SIGNATURES, name, (swapped, res))
    assert set(callers) - set(_cabi.load_callers(lib)) == {name}
    monkeypatch.setattr(_cabi, "FA_ABI_VERSION", _cabi.FA_ABI_VERSION + 1)
    assert _cabi.load_callers(lib) == {}
    assert sysconfig.get_config_var("EXT_SUFFIX") in _build.call_module_path().name
    monkeypatch.undo()
    monkeypatch.setattr(_build, "LIBDIR", tmp_path)
    _build.call_module_path().write_bytes(b"no module")
    assert _cabi.load_callers(lib) == {}


@pytest.mark.parametrize("kind", ["void_p", "byref", "bytes", "big"])
def test_what_only_ctypes_takes(both, kind, monkeypatch):
    """Arguments that ctypes resolves in its own way reach the library as through
    ctypes: a c_void_p stands for the address it holds, not for its own."""
    from frame_analytics_amd import backend

    lib, callers = both
    native = backend._Native()
    native.gpu, native.callers = lib, callers
    monkeypatch.setattr(backend, "_ext", native)
    name = "fa_gpu_ssim_once"
    buf = ctypes.create_string_buffer(64)
    p = ctypes.addressof(buf)
    n, x, k = 1, p, 4  # k = 4: refused after the pointers, before any launch
    if kind == "void_p":
        x = ctypes.c_void_p(None)  # a null pointer: refused as one
        k = 11
    elif kind == "byref":
        x = ctypes.byref(buf)
    elif kind == "bytes":
        x = bytes(64)
    else:
        n = 1 << 70  # its low bits: no image
    args = (x, p, 0, n, 1, 64, 64, None, None, None, p, k, 127.5, 6.5, 58.5, None, p, 4096,
            None, p, p, 0, None)
    want = lib.fa_gpu_ssim_once(*args)
    assert want > 0 and backend.call_gpu(name, *args) == want
    arr = memoryview(bytearray(64))  # refused by ctypes, refused still
    with pytest.raises(ctypes.ArgumentError):
        backend.call_gpu(name, arr, *args[1:])
