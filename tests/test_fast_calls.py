"""The native call paths leave every call they cannot take as it stands to
the wrappers: on the CPU, tensors that are not on a GPU."""

import importlib

import pytest
import torch

from microserve_amd import _lib


def _args(n=2, hq=4, hk=2):
    kc = torch.zeros(3, 128, hk, 128).to(torch.float8_e4m3fn)
    ks = torch.ones(3, 128, hk)
    q = torch.zeros(n, hq, 128, dtype=torch.float16)
    k = torch.zeros(n, hk, 128, dtype=torch.float16)
    i32 = torch.zeros(n, dtype=torch.int32)
    return q, k, kc, ks, i32


def test_tensors_off_the_gpu_are_left_to_the_wrappers():
    _lib.load()
    q, k, kc, ks, i32 = _args()
    f = _lib.fast
    assert f.store(k, k, kc, kc, ks, ks, i32) is None
    assert f.decode(q, kc, kc, ks, ks, i32, i32.view(-1, 1), 0.1, None, None) is None
    assert f.prefill(q, kc, kc, ks, ks, i32, None, None, 0, 2, 0, 0.1) is None
    assert f.fresh(q, k, k, i32, i32, 2, 0.1) is None
    cos = torch.ones(4, 128, dtype=torch.float16)
    assert f.prologue(i32.long(), q, k, k, None, None, 1e-6, cos, cos, kc, kc, ks, ks, i32,
                      True) is None


def test_wrong_argument_counts_and_types_are_left_to_the_wrappers():
    f = _lib.fast
    for fn in (f.store, f.decode, f.prefill, f.fresh, f.prologue):
        assert fn() is None
        assert fn(*[None] * 7) is None and fn(*["x"] * 15) is None and fn(*[3] * 10) is None


def _without_extension(monkeypatch, error):
    """A process in which importing the extension raises `error`."""
    real = importlib.import_module

    def fail(name, *a):
        if name == _lib._FAST:
            raise error
        return real(name, *a)

    monkeypatch.setattr(_lib, "_lib", None)
    monkeypatch.setattr(_lib, "fast", _lib.fast)
    monkeypatch.setattr(importlib, "import_module", fail)
    _lib.fast = _lib._import_fast()
    return real


def test_an_extension_that_does_not_load_names_its_cause(monkeypatch):
    cause = ImportError("undefined symbol: _ZN3c105ErrorE")
    _without_extension(monkeypatch, cause)
    with pytest.raises(RuntimeError, match="undefined symbol: _ZN3c105ErrorE") as e:
        _lib.fast.decode()
    assert e.value.__cause__ is cause and "not built" not in str(e.value)


def test_an_extension_built_later_is_found_by_the_next_call(monkeypatch):
    real = _without_extension(monkeypatch, ModuleNotFoundError(name=_lib._FAST))
    with pytest.raises(RuntimeError, match="not built"):
        _lib.fast.decode()
    monkeypatch.setattr(importlib, "import_module", real)
    assert _lib.fast.decode() is None
    assert _lib.fast is real(_lib._FAST)


def test_the_library_loads_without_the_extension(monkeypatch):
    _without_extension(monkeypatch, ModuleNotFoundError(name=_lib._FAST))
    assert _lib.load().mskv_version() >= 100
