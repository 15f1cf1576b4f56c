"""Calls of C functions by address (csrc/core/native_call.cpp) against ctypes: every argument arrives where the function looks for it."""
import ctypes
import random
import subprocess
from ctypes import c_float, c_int, c_longlong, c_void_p

import pytest

from llm_consensus_amd._native import core

TYPES = {"P": ("void*", c_void_p), "I": ("int", c_int), "L": ("long long", c_longlong), "F": ("float", c_float)}


def _signatures():
    rng = random.Random(3)
    out = ["", "P", "F", "IIIIII", "IIIIIII", "FIFIFIFIF"[:8], "P" * 16, "P" * 17, "L" * 32 + "I", "I" * 48 + "F" * 8]
    for _ in range(20):
        n = rng.randint(1, 40)
        s = [rng.choice("PIL") for _ in range(n)]
        for i in rng.sample(range(n), min(n, rng.randint(0, 8))):
            s[i] = "F"
        out.append("".join(s))
    return out


@pytest.fixture(scope="module")
def echoes(tmp_path_factory):
    """For every signature a function that writes its arguments, as doubles, into ``echoed`` and returns minus their number."""
    d = tmp_path_factory.mktemp("native_call")
    src = "extern double echoed[64];\ndouble echoed[64];\n"
    sigs = _signatures()
    for k, s in enumerate(sigs):
        params = ", ".join(f"{TYPES[c][0]} a{i}" for i, c in enumerate(s)) or "void"
        body = "".join(f"echoed[{i}] = (double)({'long long' if c == 'P' else TYPES[c][0]})a{i}; " for i, c in enumerate(s))
        src += f"int echo{k}({params}) {{ {body}return -{len(s)}; }}\n"
    (d / "echo.c").write_text(src)
    subprocess.run(["gcc", "-O2", "-shared", "-fPIC", "-o", str(d / "echo.so"), str(d / "echo.c")], check=True)
    return ctypes.CDLL(str(d / "echo.so")), sigs


def test_arguments_arrive(echoes):
    lib, sigs = echoes
    seen = (ctypes.c_double * 64).in_dll(lib, "echoed")
    rng = random.Random(5)
    for k, s in enumerate(sigs):
        fn = getattr(lib, f"echo{k}")
        fn.argtypes, fn.restype = [TYPES[c][1] for c in s], c_int
        fast = core.native_call(ctypes.cast(fn, c_void_p).value, s, f"echo{k}")
        pools = {"P": [None, 0, 1 << 47, 4096], "I": [0, -1, -2**31, 2**31 - 1, True], "L": [0, -1, 2**52, -2**52], "F": [0.0, -1.5, 0.1, 3e38]}
        for _ in range(4):
            args = [rng.choice(pools[c]) for c in s]
            fn(*args)
            want = list(seen[:len(s)])
            seen[:] = [7.0] * 64
            assert fast(*args) == -len(s)
            assert list(seen[:len(s)]) == want, s


def test_other_arguments_are_left_to_the_general_way(echoes):
    lib, sigs = echoes
    k = sigs.index("FIFIFIFI")
    fast = core.native_call(ctypes.cast(getattr(lib, f"echo{k}"), c_void_p).value, sigs[k], "echo")
    good = [1.0, 2] * 4
    assert fast(*good) == -8
    for i, bad in ((0, 1), (0, None), (1, None), (1, 2.0), (1, "2")):
        assert fast(*good[:i], bad, *good[i + 1:]) is NotImplemented
    assert fast(*good[:7]) is NotImplemented and fast(*good, 1) is NotImplemented
    for address, kinds in ((0, "I"), (1, "X"), (1, "F" * 9), (1, "I" * 49)):
        with pytest.raises(ValueError):
            core.native_call(address, kinds, "f")
