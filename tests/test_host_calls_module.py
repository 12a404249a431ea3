"""CPU: the Python module over the library's entry points and the library belong to one header, and between them lack nothing."""

import types

import pytest

import keras_amd
from keras_amd import _k3q_calls, _lib


def test_every_entry_point_has_its_place():
    names = {n for n in dir(_k3q_calls) if n.startswith("k3q_")}
    assert names == set(_lib.SIGNATURES) - _lib.BY_CTYPES
    calls = _lib.calls()
    for name in _lib.SIGNATURES:
        assert isinstance(getattr(calls, name), types.BuiltinFunctionType) == (name not in _lib.BY_CTYPES)


@pytest.mark.parametrize("change", ["digest", "no digest", "name"])
def test_a_module_of_another_build_is_refused(monkeypatch, change):
    other = types.SimpleNamespace(**{n: getattr(_k3q_calls, n) for n in dir(_k3q_calls) if not n.startswith("__")})
    if change == "digest":
        other.header_digest = "0" * 16
    elif change == "no digest":
        del other.header_digest
    else:
        del other.k3q_gemm_i8
    monkeypatch.setattr(keras_amd, "_k3q_calls", other)
    with pytest.raises(AttributeError if change == "name" else RuntimeError):
        _lib._Calls(_lib.load())
