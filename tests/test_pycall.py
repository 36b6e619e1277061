"""The direct Python callables of the hot entry points hand over what ctypes hands over, and leave everything else to it."""
import ctypes as C
import types

import numpy as np
import pytest

import skainet_amd
from skainet_amd import build, runtime

pycall = pytest.importorskip("skainet_amd._pycall")

_V, _I = C.c_void_p, C.c_int
SIGNATURES = {"matvec_q": [_V, _I, _V, _I, _I, _V, _V], "gemm_q": [_V, _I, _V, _I, _I, _V, _I, _V],
              "attn_decode": [_V, _V, _V, C.POINTER(C.c_int32), C.c_float, _V]}
CASES = {
    "matvec_q": [(1, 12, 2, 3, 4, 5, 6), (2**48 + 16, 14, 2**63 + 32, -1, 2**31 - 1, 2**64 - 16, 0), (-16, 12, 2**64 + 16, 2**32 + 7, -2**31, 1, 1),
                 (1, np.int64(12), np.int64(64), 3, 4, None, 6), (1, True, 2, 3, 4, 5, 6)],
    "gemm_q": [(1, 8, 2, 3, 4, 5, 6, 7), (2**48, 13, 2**63, -5, 2**33 + 1, 2**50, 2**40, 2**62), (1, 8, None, 3, 4, 5, 6, 7)],
    "attn_decode": [(1, 2, 3, None, 0.0883883, 4), (2**48, 2**63, 2**50, None, 1e-50, 0), (1, 2, 3, (C.c_int32 * 2)(7, 9), 0.5, 4), (1, 2, 3, None, 1, 4)],
}


@pytest.mark.parametrize("name,args", [(n, a) for n in CASES for a in CASES[n]])
def test_the_arguments_arrive_as_through_ctypes(name, args):
    seen = []

    def record(*a):
        seen.append(tuple(None if v is None else v[0:2] if isinstance(v, C.POINTER(C.c_int32)) and v else float(v) if isinstance(v, float) else
                          None if isinstance(v, C.POINTER(C.c_int32)) else v for v in a))
        return -7

    fn = C.CFUNCTYPE(C.c_int, *SIGNATURES[name])(record)
    lib = runtime.load_library()

    def general(*a):
        return fn(*[runtime._ptr(v) if t is _V else v for v, t in zip(a, SIGNATURES[name])])

    at = C.cast(fn, C.c_void_p).value
    library_at = C.cast(getattr(lib, "skn_" + name), C.c_void_p).value
    try:
        pycall.bind(name, at, general)
        assert getattr(pycall, name)(*args) == -7
        assert general(*args) == -7
    finally:
        pycall.bind(name, library_at, _GENERAL[name])
    assert seen[0] == seen[1]


def _refuse(*_):
    raise TypeError("the general call")


@pytest.mark.parametrize("name,args", [("matvec_q", (1, 12, 2, 3, 4, 5)), ("matvec_q", (1, 12.0, 2, 3, 4, 5, 6)), ("gemm_q", (1, 12, "w", 3, 4, 5, 6, 7)),
                                       ("attn_decode", (1, 2, 3, [4], 0.5, 5))])
def test_other_arguments_go_to_the_general_call(name, args):
    lib = runtime.load_library()
    library_at = C.cast(getattr(lib, "skn_" + name), C.c_void_p).value
    try:
        pycall.bind(name, library_at, _refuse)
        with pytest.raises(TypeError, match="the general call"):
            getattr(pycall, name)(*args)
    finally:
        pycall.bind(name, library_at, _GENERAL[name])


def _matvec(handle, ggml_type, w, n, k, x, y):
    return runtime.load_library().skn_matvec_q(handle, ggml_type, runtime._ptr(w), n, k, runtime._ptr(x), runtime._ptr(y))


def _gemm(handle, ggml_type, w, n, k, a, m, c):
    return runtime.load_library().skn_gemm_q(handle, ggml_type, runtime._ptr(w), n, k, runtime._ptr(a), m, runtime._ptr(c))


def _attn(handle, kv, q, n_ctx, scale, out):
    return runtime.load_library().skn_attn_decode(handle, kv, runtime._ptr(q), n_ctx, scale, runtime._ptr(out))


_GENERAL = {"matvec_q": _matvec, "gemm_q": _gemm, "attn_decode": _attn}


def test_a_second_load_binds_the_same_general_calls(monkeypatch):
    """Two threads may both load the library first: the callable that is bound second must not get itself as its general call, which it
    would then call without end."""
    bound = []
    lib = runtime.load_library()
    fake = types.SimpleNamespace(bind=lambda name, at, general: bound.append((name, general)), matvec_q=len, gemm_q=len, attn_decode=len)
    monkeypatch.setattr(skainet_amd, "_pycall", fake)
    for name in SIGNATURES:
        monkeypatch.setattr(runtime, "_" + name, getattr(runtime, "_" + name))  # (put back afterwards)
    for _ in range(2):
        runtime._bind_direct(lib, runtime.LIB_PATH)
    assert len(bound) == 6 and bound[:3] == bound[3:]
    assert all(isinstance(general, types.FunctionType) for _, general in bound)


@pytest.mark.parametrize("stop", ["compiler fails", "no compiler"])
def test_the_library_is_built_without_them_where_they_cannot_be(monkeypatch, tmp_path, capsys, stop):
    target = tmp_path / "_pycall.so"
    target.write_bytes(b"of older sources")
    monkeypatch.setattr(build, "PYCALL", str(target))
    if stop == "no compiler":
        monkeypatch.setattr(build.shutil, "which", lambda name: None)
    else:
        cc = tmp_path / "cc"
        cc.write_text("#!/bin/sh\necho no space left\nexit 1\n")
        cc.chmod(0o755)
        monkeypatch.setattr(build.shutil, "which", lambda name: str(cc))
    build.build_pycall()
    assert not target.exists()
    assert ("no space left" if stop == "compiler fails" else "no C compiler") in capsys.readouterr().err
