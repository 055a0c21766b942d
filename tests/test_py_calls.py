"""The Python functions of a step's entry points (csrc/py_calls.cpp) pass what ctypes passes for the same prototypes, and
refuse what it refuses."""
import ctypes as C
import random

import pytest

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
