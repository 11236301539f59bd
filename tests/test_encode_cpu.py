"""The binding's per-operator call (ksearch_amd/pyext/encode.c) and its ctypes form hand the library the same arguments and
accept and refuse the same ones; without the extension the library still loads.  A recording function stands in for
ksh_encode; no GPU work."""
import ctypes as C
import subprocess
import sys

import numpy as np
import pytest

from ksearch_amd import hip

PROTO = C.CFUNCTYPE(C.c_int, C.c_void_p, C.c_void_p, C.POINTER(C.c_void_p), C.POINTER(C.c_uint64), C.c_int, C.POINTER(C.c_void_p),
                    C.POINTER(C.c_uint64), C.c_int)


class Buf:
    def __init__(self, h):
        self.h = h


@pytest.fixture(params=["extension", "ctypes"])
def call(request, monkeypatch):
    seen = []

    def fn(ctx, kernel, ins, in_off, n_in, outs, out_off, n_out):
        def side(p, off, n):
            return [(p[i], off[i] if off else 0) for i in range(min(n, 8))]
        seen.append((ctx, kernel, n_in, side(ins, in_off, n_in), n_out, side(outs, out_off, n_out)))
        return 7

    keep = PROTO(fn)
    hip.lib()
    if request.param == "ctypes":
        monkeypatch.setattr(hip, "ENCODE_PATH", "/nonexistent/_encode.so")
    encode = hip._load_encode(keep)
    assert (type(encode).__name__ == "function") == (request.param == "ctypes")
    yield lambda *a: (encode(*a), seen.pop())
    hip._load_encode(hip.lib().ksh_encode)       # (the extension keeps one address)


def test_arguments_reach_the_library(call):
    a, b, c = Buf(0x1000), Buf(0xFFFF_FFFF_FFFF_F000), Buf(None)
    want = (0x11, 0x22, 2, [(0x1000, 0), (0xFFFF_FFFF_FFFF_F000, 0)], 1, [(0x1000, 0)])
    for ins in ([a, b], (a, b), (x for x in (a, b))):
        assert call(0x11, 0x22, ins, None, [a], None) == (7, want)
    # offsets: fewer than bindings, numpy numbers, whatever int() takes, no kernel and a null binding
    assert call(None, None, [a, c], [16], (b,), (np.int64(1 << 40),)) == (
        7, (None, None, 2, [(0x1000, 16), (None, 0)], 1, [(0xFFFF_FFFF_FFFF_F000, 1 << 40)]))
    assert call(1, 2, [a], [32.0], [], None)[1] == (1, 2, 1, [(0x1000, 32)], 0, [])
    # more bindings than any kernel has: the library's to refuse
    assert call(1, 2, [a] * 40, None, [b] * 17, [4] * 17)[1][2::2] == (40, 17)


def test_refusals(call):
    a = Buf(0x1000)
    with pytest.raises(IndexError):
        call(1, 2, [a], [1, 2], [a], None)
    with pytest.raises(AttributeError):
        call(1, 2, [object()], None, [a], None)
    with pytest.raises(TypeError):
        call(1, 2, [a], ["x", None][1:], [a], None)
    with pytest.raises(TypeError):
        call(1, 2, 5, None, [a], None)


def test_the_library_loads_without_the_extension():
    code = "from ksearch_amd import hip; hip.ENCODE_PATH = '/nonexistent'; hip.lib(); print(type(hip._encode).__name__)"
    r = subprocess.run([sys.executable, "-c", code], capture_output=True, text=True, cwd=str(hip._HERE) + "/..")
    assert r.returncode == 0 and r.stdout.strip() == "function", r.stderr
