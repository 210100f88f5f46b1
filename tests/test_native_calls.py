"""The entry points as native callables: what the library is given is what ctypes would have given it."""
import ctypes
import os
import shutil
import sysconfig
from ctypes import c_float, c_int, c_long, c_void_p

import pytest

from axon_amd.kernels import build, lib

calls = lib._calls_module()
needs = pytest.mark.skipif(not os.path.exists(os.path.join(sysconfig.get_paths()["include"], "Python.h")) or shutil.which("g++") is None,
                           reason="no headers of this Python, or no compiler: the calls go through ctypes")


def bound(name, restype, argtypes):
    seen = []

    def entry(*args):
        seen.append(args)
        return 7
    made = ctypes.CFUNCTYPE(restype, *argtypes)(entry)
    return calls.bind(name, ctypes.cast(made, c_void_p).value), seen, made


@needs
def test_every_signature_has_its_callable():
    assert set(lib._SIGNATURES) <= set(calls.names())
    for name, argtypes in lib._SIGNATURES.items():
        fn, seen, _ = bound(name, c_int, argtypes)
        with pytest.raises(TypeError):
            fn(*[0] * (len(argtypes) + 1))                # as many arguments as the header declares
        assert fn(*[0] * len(argtypes)) == 7 and len(seen) == 1
    with pytest.raises(KeyError):
        calls.bind("axk_nothing", 1)


@needs
def test_arguments_arrive():
    fn, seen, _ = bound("axk_add_scaled", c_int, lib._SIGNATURES["axk_add_scaled"])       # pointer, pointer, float, long, pointer
    high = 0x7fff_1234_5678_9abc
    assert fn(high, None, 0.1, 1 << 40, c_void_p(4096)) == 7
    assert fn(0, c_void_p(None), 3, -5, high) == 7
    assert seen == [(high, None, ctypes.c_float(0.1).value, 1 << 40, 4096), (None, None, 3.0, -5, high)]
    fn, seen, _ = bound("axk_gemm_workspace", c_long, [c_int] * 4)
    assert fn(-1, True, 1 << 31, 2 ** 31 - 1) == 7 and seen == [(-1, 1, -(1 << 31), 2 ** 31 - 1)]


@needs
@pytest.mark.parametrize("args", [(1, 2, 3.0, 4), (1.5, 2, 3.0, 4, 5), ("a", 2, 3.0, 4, 5), (1, 2, None, 4, 5), (1, 2, 3.0, 4.5, 5), (1, 2, 3.0, 1 << 70, 5)])
def test_what_is_no_number_or_address_is_refused(args):
    fn, seen, _ = bound("axk_add_scaled", c_int, [c_void_p, c_void_p, c_float, c_long, c_void_p])
    with pytest.raises((TypeError, AttributeError, OverflowError)):
        fn(*args)
    assert not seen


@needs
def test_kinds_of_arguments_are_those_of_the_signatures():
    """A number with a fraction is taken where ctypes is told of a float, None where it is told of an address."""
    for name, argtypes in lib._SIGNATURES.items():
        fn, _, _made = bound(name, c_int, argtypes)
        for i, kind in enumerate(argtypes):
            for value, fits in ((1.5, kind is c_float), (None, kind is c_void_p)):
                args = [0] * len(argtypes)
                args[i] = value
                if fits:
                    assert fn(*args) == 7
                else:
                    with pytest.raises((TypeError, AttributeError)):
                        fn(*args)


@pytest.mark.parametrize("error", [build.MissingError("no Python.h"), build.BuildError("compiling axon_calls failed"), ImportError("a symbol"),
                                   PermissionError("a folder that cannot be written")])
def test_without_native_calls_ctypes_goes_on_and_a_line_says_so(error, monkeypatch, capsys):
    def build_calls(force=False):
        raise error
    monkeypatch.setattr(build, "build_calls", build_calls)
    monkeypatch.setattr(lib, "_calls", False)
    assert lib._calls_module() is None and lib._calls_module() is None
    said = capsys.readouterr().err
    assert said.count("ctypes") == 1 and str(error) in said


def test_a_build_of_everything_stops_at_calls_that_do_not_compile(monkeypatch):
    made = []
    for name in ("build_host", "build_kernels"):
        monkeypatch.setattr(build, name, lambda *a: made.append(a))
    for error, passes in ((build.MissingError("no Python.h"), True), (build.BuildError("an error"), False)):
        def build_calls(force=False, error=error):
            raise error
        monkeypatch.setattr(build, "build_calls", build_calls)
        if passes:
            assert len(build.build_all()) == 3
        else:
            with pytest.raises(build.BuildError, match="an error"):
                build.build_all()
