"""The serving binding's bytes objects -- independent of what other modules
make of ctypes.pythonapi, which it leaves alone, and never handed out unless
the library filled them."""
import ctypes as C
import os
import subprocess
import sys

import pytest

import serving as S

PKG = os.path.dirname(os.path.abspath(S.__file__))
DATA = bytes(range(256)) * 3 + b"\0\0\1"


class _Lib:
    """rvs_server_output of one kept output, whose second call sees `again`."""

    def __init__(self, again=DATA):
        self.again = again

    def rvs_server_output(self, h, k, out, cap):
        if out is None:
            return len(DATA)
        assert type(out) is int, "not the address of the new object"
        C.memmove(out, self.again, min(cap, len(self.again)))
        return len(self.again) or -1

    def rvs_server_destroy(self, h):
        pass


def _output(monkeypatch, lib):
    monkeypatch.setattr(S, "_lib", lambda: lib)
    srv = S.Server.__new__(S.Server)
    srv.h = 1
    return srv.output(0)


def test_output_whatever_others_declare(monkeypatch):
    """Another module's prototypes of the interpreter's functions do not reach this one's."""
    monkeypatch.setattr(C.pythonapi.PyBytes_AsString, "restype", C.c_char_p)
    assert _output(monkeypatch, _Lib()) == DATA


def test_import_leaves_the_shared_functions_alone():
    code = ("import ctypes as C, serving; f = C.pythonapi.PyBytes_AsString; f.restype = C.c_char_p; "
            "assert f.argtypes is None and f(C.py_object(b'abc')) == b'abc'; "
            "assert C.pythonapi.PyBytes_FromStringAndSize.argtypes is None")
    subprocess.run([sys.executable, "-c", code], check=True, env=dict(os.environ, PYTHONPATH=PKG))


@pytest.mark.parametrize("again", [b"", DATA[:100], DATA + b"x"], ids=["gone", "shorter", "longer"])
def test_output_that_changed_is_refused(monkeypatch, again):
    with pytest.raises(RuntimeError):
        _output(monkeypatch, _Lib(again))


@pytest.mark.gpu
@pytest.mark.parametrize("keep", [False, True])
def test_outputs_that_are_not_kept(torch_cuda, keep):
    print("case outputs, kept %d" % keep, flush=True)
    import workloads as W
    rg = W.rig("rects_640", scale=4)
    src = W.device_sources(rg, W.render_sources(rg))
    srv = S.Server([src], memory_budget=1 << 30, max_batch=2, slots=1, keep_outputs=keep)
    try:
        srv.run_closed([(0, W.device_target(rg))] * 2, 2)
        if keep:
            assert len(srv.output(1)) > 0
        for k in (2, -1) if keep else (0, 1):
            with pytest.raises(RuntimeError):
                srv.output(k)
    finally:
        srv.close()
