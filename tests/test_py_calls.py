"""The Python functions of a step's entry points (csrc/py_calls.cpp) pass what ctypes passes for the same prototypes, and
refuse what it refuses."""
import ctypes as C
import random
import warnings

import numpy as np
import pytest
import torch

from gllm_amd import _calls
from gllm_amd.backend import load_library, step_calls


def receiver(argtypes, rc):
    seen = []
    proto = C.CFUNCTYPE(C.c_int, *[C.c_void_p if isinstance(t, type) and issubclass(t, C._Pointer) else t for t in argtypes])
    fn = proto(lambda *a: seen.append(a) or rc)
    return fn, C.cast(fn, C.c_void_p).value, seen


def value(t, rng):
    if t is C.c_float:
        return rng.choice([0.1, -2.5, 1, 3.0e38])
    if t is C.c_void_p:
        return rng.choice([None, 1, 2 ** 47 + 12345, 2 ** 64 - 16])
    return rng.choice([0, 1, 12, 2 ** 31 - 1, 2 ** 32 + 5, 2 ** 63, -1, True])


@pytest.mark.parametrize("name", _calls.names)
def test_arguments_arrive_as_through_ctypes(name):
    argtypes = [C.c_void_p if isinstance(t, type) and issubclass(t, C._Pointer) else t for t in getattr(load_library(), name).argtypes]
    rng = random.Random(name)
    for _ in range(50):
        rc = rng.choice([0, 1, 5, -3])
        fn, address, seen = receiver(argtypes, rc)
        args = [value(t, rng) for t in argtypes]
        assert _calls.bind(name, address)(*args) == rc
        assert C.CFUNCTYPE(C.c_int, *argtypes)(address)(*args) == rc
        assert seen[0] == seen[1]


@pytest.mark.parametrize("name", _calls.names)
def test_refuses_what_ctypes_refuses(name):
    argtypes = [C.c_void_p if isinstance(t, type) and issubclass(t, C._Pointer) else t for t in getattr(load_library(), name).argtypes]
    fn, address, seen = receiver(argtypes, 0)
    call, good = _calls.bind(name, address), [1.0 if t is C.c_float else 1 for t in argtypes]
    for i, t in enumerate(argtypes):
        for bad in ("1", [], object()) if t is C.c_float else (1.0, [], object()) if t is C.c_void_p else (1.0, "1", None):
            with pytest.raises(C.ArgumentError):
                call(*good[:i], bad, *good[i + 1:])
    for args in (good[:-1], good + [1], []):
        with pytest.raises(TypeError):
            call(*args)
    assert not seen


def test_bound_to_the_loaded_library():
    lib, calls = load_library(), step_calls()
    assert set(calls) == set(_calls.names)
    # without a context every entry point answers with a status and touches nothing
    assert calls["gllmq_quantized_matmul_ex"](None, None, 0, None, None, 12, 1, 1, 256, 0, None) == \
        lib.gllmq_quantized_matmul_ex(None, None, 0, None, None, 12, 1, 1, 256, 0, None) != 0
    with pytest.raises(KeyError):
        _calls.bind("gllmq_nothing", 1)


class Index:
    def __index__(self):
        return 2 ** 33 + 6


class Parameter:
    _as_parameter_ = 9


def through(fn, args, seen):
    """What arrives, or that it is refused."""
    seen.clear()
    try:
        with warnings.catch_warnings():
            warnings.simplefilter("ignore")
            rc = fn(*args)
    except Exception as e:
        assert not seen
        return type(e)
    return rc, seen[0]


@pytest.mark.parametrize("name", _calls.names)
def test_whatever_ctypes_takes_or_refuses(name):
    """Integers of numpy's, torch scalars, ctypes objects, anything that says what it is as an index or a parameter, and what is none of
    those: accepted with the same value as through ctypes, or refused with the same exception."""
    argtypes = [C.c_void_p if isinstance(t, type) and issubclass(t, C._Pointer) else t for t in getattr(load_library(), name).argtypes]
    fn, address, seen = receiver(argtypes, 3)
    call, plain = _calls.bind(name, address), C.CFUNCTYPE(C.c_int, *argtypes)(address)
    good = [1.0 if t is C.c_float else 1 for t in argtypes]
    values = [np.int64(5), np.uint32(7), np.int8(-1), np.bool_(True), np.float32(2.5), np.array(3), np.zeros(2, np.int64), torch.tensor(3), torch.tensor(3.5),
              torch.tensor([1, 2]), C.c_size_t(2 ** 40), C.c_uint32(4), C.c_int(-4), C.c_float(4.5), C.c_void_p(2 ** 40), C.c_void_p(None), Index(), Parameter(),
              2 ** 70, -1, None, True, 1.5, 3, "a", [], object()]
    accepted = 0
    for i, t in enumerate(argtypes):
        for v in values:
            if isinstance(v, str) and t is C.c_void_p:
                continue  # (a pointer to a copy of the text, which differs from call to call)
            args = good[:i] + [v] + good[i + 1:]
            got, want = through(call, args, seen), through(plain, args, seen)
            assert got == want, (i, t, v)
            accepted += isinstance(got, tuple)
    assert accepted > 6 * len(argtypes)


def test_without_the_module(monkeypatch):
    """The backend's calls are there, with the same results, where the module was not built."""
    import sys
    from gllm_amd import backend
    want = backend.step_calls()["gllmq_moe_route"](None, None, 1, 1, 1, 1.0, None, None, None, None, None, None, None)
    monkeypatch.setattr(backend, "_step_calls", None)
    monkeypatch.setitem(sys.modules, "gllm_amd._calls", None)
    monkeypatch.delattr("gllm_amd._calls")
    calls = backend.step_calls()
    assert set(calls) == set(_calls.names) and not any(type(fn) is type(_calls.bind) for fn in calls.values())
    assert calls["gllmq_moe_route"](None, None, 1, 1, 1, 1.0, None, None, None, None, None, None, None) == want != 0
    arr = (backend.MatmulDesc * 1)()
    assert calls["gllmq_quantized_matmul_batch"](None, C.addressof(arr), 1, None) != 0
