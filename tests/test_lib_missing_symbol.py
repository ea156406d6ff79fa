"""A library of the same ABI version that lacks an entry point of the binding (built before it was
added) is refused with the name and the advice to rebuild, not with an attribute error."""

import ctypes

import pytest

from giwaxsim_amd import _lib


class _Older:
    """The loaded library without one symbol."""

    def __init__(self, lib, missing):
        self._lib, self._missing = lib, missing

    def __getattr__(self, name):
        if name == self._missing:
            raise AttributeError(f"undefined symbol: {name}")
        return getattr(self._lib, name)


def test_named_error(monkeypatch):
    real = ctypes.CDLL(_lib.LIB)
    monkeypatch.setattr(_lib, '_lib', None)
    monkeypatch.setattr(ctypes, 'CDLL', lambda path: _Older(real, 'gx_detector_work_size'))
    with pytest.raises(_lib.GxError, match='gx_detector_work_size.*rebuild'):
        _lib.load()


def test_version_comes_first(monkeypatch):
    """A library of another version is refused for that, whatever it lacks."""
    real = ctypes.CDLL(_lib.LIB)
    older = _Older(real, 'gx_detector_work_size')
    older.gx_abi_version = ctypes.CFUNCTYPE(ctypes.c_int)(lambda: _lib.GX_ABI_VERSION - 1)
    monkeypatch.setattr(_lib, '_lib', None)
    monkeypatch.setattr(ctypes, 'CDLL', lambda path: older)
    with pytest.raises(_lib.GxError, match='ABI version'):
        _lib.load()
