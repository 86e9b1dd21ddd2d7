"""The native way to an entry point (csrc/calls.cpp) beside ctypes: the same values arrive whatever the order of integers, pointers
and floats, and what it does not take itself ctypes takes or refuses."""
import ctypes
import subprocess
from ctypes import c_float, c_int, c_int64, c_void_p

import pytest

from mini_engine_amd.kernels import build, ops

SOURCE = r'''
#include <cstdio>
#include <cstring>
static char said[512];
extern "C" const char* me_last_error() { return said; }
extern "C" int me_mixed(void* a, long b, int c, float d, int e, int f, int g, int h, int i, float j, long k, int rc, void* l, float m) {
  snprintf(said, sizeof said, "%p %ld %d %g %d %d %d %d %d %g %ld %p %g", a, b, c, d, e, f, g, h, i, j, k, l, m);
  return rc;
}
extern "C" int me_many(float a, long b0, long b1, long b2, long b3, long b4, long b5, long b6, long b7, long b8, long b9, float c, float d, float e,
                       float f, float g, float h, float i, int last) {
  snprintf(said, sizeof said, "%g %ld %ld %g %g %d", a, b0, b9, c, i, last);
  return 1;
}
extern "C" int me_none() { strcpy(said, "none"); return 0; }
'''
P, I, L, F = c_void_p, c_int, c_int64, c_float
PROTOS = {"me_mixed": [P, L, I, F, I, I, I, I, I, F, L, I, P, F], "me_many": [F] + [L] * 10 + [F] * 7 + [I], "me_none": []}


@pytest.fixture(scope="module")
def library(tmp_path_factory):
    path = tmp_path_factory.mktemp("calls") / "libentries.so"
    (path.parent / "entries.cpp").write_text(SOURCE)
    subprocess.run(["g++", "-O2", "-shared", "-fPIC", str(path.parent / "entries.cpp"), "-o", str(path)], check=True)
    return str(path)


def test_every_argument_arrives_as_ctypes_passes_it(library):
    if ops._native_calls() is None:
        pytest.skip("no headers of Python here: the entry points are called through ctypes")
    lib, plain = ops._Lib(library, PROTOS), ctypes.CDLL(library)
    assert type(lib.fns["me_mixed"]).__module__ == "me_calls"
    said = lambda: lib.cdll.me_last_error().decode()
    for args in ((None, -5, 7, 1.5, -1, 2, 3, 4, 5, 2.25, 1 << 40, 0, 140000000000000, -3.0), (0, 1 << 62, -(1 << 31), 0.0, True, 2, 3, 4, 5, -1e30, -1, 0, None, 1e-3)):
        lib.call("me_mixed", *args)
        ours = said()
        fn = plain.me_mixed
        fn.argtypes, fn.restype = PROTOS["me_mixed"], c_int
        assert fn(*args) == 0 and said() == ours
    lib.call("me_none")
    assert said() == "none"
    many = (0.5, *range(10), 1.0, 2.0, 3.0, 4.0, 5.0, 6.0, 7.0, -9)
    with pytest.raises(ops.KernelError, match="me_many: 0.5 0 9 1 7 -9"):
        lib.call("me_many", *many)
    assert lib.fns["me_many"](*many) == 1


def test_what_is_no_plain_number_goes_to_ctypes(library):
    lib = ops._Lib(library, PROTOS)
    good = (None, -5, 7, 1.5, -1, 2, 3, 4, 5, 2.25, 9, 0, 12, -3.0)
    lib.call("me_mixed", (c_void_p * 2)(), *good[1:])                                # an array stands for its address
    lib.call("me_mixed", *good[:3], 1, *good[4:])                                    # an integer for a float
    for bad in (good[:-1], good[:1] + (None,) + good[2:], good[:2] + (1.5,) + good[3:]):
        with pytest.raises((TypeError, ctypes.ArgumentError)):
            lib.call("me_mixed", *bad)
    with pytest.raises(KeyError):
        lib.call("me_unknown")


@pytest.fixture()
def fresh(monkeypatch, tmp_path):
    """A folder of libraries of its own in which nothing is built, and no module kept from before."""
    monkeypatch.setattr(build, "PKG_LIB", str(tmp_path / "lib"))
    monkeypatch.setattr(build, "_fallback", str(tmp_path / "none"))
    (tmp_path / "lib").mkdir()
    ops._native_calls.cache_clear()
    yield tmp_path
    ops._native_calls.cache_clear()


def _compiler(tmp_path, line):
    path = tmp_path / "hipcc"
    path.write_text(f"#!/bin/sh\n{line}\n")
    path.chmod(0o755)
    return str(path)


@pytest.mark.parametrize("why", ["does not compile", "cannot be loaded", "another machine", "no compiler"])
def test_without_the_module_the_entry_points_are_called_through_ctypes(monkeypatch, fresh, library, why):
    if why == "another machine":
        monkeypatch.setattr(build.platform, "machine", lambda: "aarch64")
    # (what "links" writes is no library)
    lines = {"does not compile": "echo no headers >&2; exit 1", "cannot be loaded": 'while [ $# -gt 1 ]; do [ "$1" = -o ] && echo x > "$2"; shift; done'}
    monkeypatch.setattr(build, "hipcc_path", lambda: None if why == "no compiler" else _compiler(fresh, lines.get(why, "exit 1")))
    assert build.calls_module() is None
    lib = ops._Lib(library, PROTOS)
    lib.call("me_none")
    assert isinstance(lib.fns["me_none"], ctypes._CFuncPtr)
    with pytest.raises(ops.KernelError, match="me_many: 0.5 0 9 1 7 -9"):
        lib.call("me_many", 0.5, *range(10), 1.0, 2.0, 3.0, 4.0, 5.0, 6.0, 7.0, -9)
