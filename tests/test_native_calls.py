"""The C ABI's Python calls (binding/calls.cpp) convert every argument as ctypes does, and step aside where they cannot."""
import ctypes
import os
import subprocess
import sysconfig

import pytest

from sglang_amd import build, native

HEADER = """#include <stdint.h>
#ifdef __cplusplus
extern "C" {
#endif
int echo(int64_t* out, const void* p, int64_t a, int b, float c, int64_t d, int e, float f, const int32_t* q, uint8_t* r, int64_t s, int t, int u);
int64_t wide(int64_t a);
int absent(int a);
const char* text(void);
#ifdef __cplusplus
}
#endif
"""
SOURCE = """#include "sglang_amd.h"
#include <string.h>
int echo(int64_t* out, const void* p, int64_t a, int b, float c, int64_t d, int e, float f, const int32_t* q, uint8_t* r, int64_t s, int t, int u) {
  int32_t ci, fi;
  memcpy(&ci, &c, 4); memcpy(&fi, &f, 4);
  int64_t v[12] = {(int64_t)p, a, b, ci, d, e, fi, (int64_t)q, (int64_t)r, s, t, u};
  memcpy(out, v, sizeof(v));
  return 7;
}
int64_t wide(int64_t a) { return a - 1; }
const char* text(void) { return "text"; }
"""


@pytest.fixture(scope="module")
def both(tmp_path_factory):
    d = tmp_path_factory.mktemp("calls")
    (d / "sglang_amd.h").write_text(HEADER.replace("int echo", "int sgl_amd_echo").replace("wide", "sgl_amd_wide").replace("absent", "sgl_amd_absent")
                                    .replace("text(", "sgl_amd_text("))
    (d / "lib.c").write_text(SOURCE.replace("int echo", "int sgl_amd_echo").replace("wide", "sgl_amd_wide").replace("* text", "* sgl_amd_text"))
    subprocess.run([build._hipcc(), "-x", "c", "-shared", "-fPIC", f"-I{d}", str(d / "lib.c"), "-o", str(d / "lib.so")], check=True)
    if build.build_calls(d / "_calls.so", d / "sglang_amd.h") is None:
        pytest.skip("no Python headers")
    cdll = ctypes.CDLL(str(d / "lib.so"))
    for name, (ret, args) in native.parse_header(d / "sglang_amd.h").items():
        if name != "sgl_amd_absent":
            getattr(cdll, name).argtypes, getattr(cdll, name).restype = args, {"int": ctypes.c_int, "int64_t": ctypes.c_int64}.get(ret, ctypes.c_char_p)
    with pytest.MonkeyPatch.context() as m:
        m.setattr(native, "CALLS_PATH", d / "_calls.so")
        assert native._load_calls(d / "lib.so") == {}                  # (another header than the one it was built for)
        m.setattr(native, "HEADER_PATH", d / "sglang_amd.h")
        calls = native._load_calls(d / "lib.so")
    return calls, cdll


def test_arguments_are_those_of_ctypes(both):
    calls, cdll = both
    for args in ((None, 1, 2, 3.5, 4, 5, 6.25, None, 0, 7, 8, 9), (2 ** 63 + 5, -2 ** 63, -1, 1, 2 ** 63 - 1, True, False, 2 ** 47, 2 ** 64 - 1, -3, -2 ** 31, 2 ** 31 - 1),
                 (0, 2 ** 64 + 3, 2 ** 32 + 9, 1e300, -2 ** 70, 2 ** 31, 1e-60, 1, 2, 0, -2 ** 33 - 1, 0), (1, 0, 0, float("nan"), 0, 0, float("-inf"), None, None, 0, 0, 0)):
        got, want = (ctypes.c_int64 * 12)(), (ctypes.c_int64 * 12)()
        assert calls["sgl_amd_echo"](ctypes.addressof(got), *args) == 7 and cdll.sgl_amd_echo(ctypes.addressof(want), *args) == 7
        assert list(got) == list(want), args
    assert calls["sgl_amd_wide"](-2 ** 62) == cdll.sgl_amd_wide(-2 ** 62) == -2 ** 62 - 1


def test_what_is_left_to_ctypes(both):
    calls, _ = both
    assert "sgl_amd_absent" not in calls
    assert calls["sgl_amd_text"]() is NotImplemented                        # (no number comes back)
    assert calls["sgl_amd_wide"]() is NotImplemented and calls["sgl_amd_wide"](1, 2) is NotImplemented
    for odd in (1.5, "1", None, ctypes.c_int64(3)):
        assert calls["sgl_amd_wide"](odd) is NotImplemented
    buf = (ctypes.c_int64 * 12)()
    assert calls["sgl_amd_echo"](ctypes.byref(buf), *([0] * 12)) is NotImplemented and calls["sgl_amd_echo"](0, 1.0, *([0] * 11)) is NotImplemented


def test_another_interpreters_module_is_not_looked_at():
    assert native.CALLS_PATH.name == "_calls" + sysconfig.get_config_var("EXT_SUFFIX") and sysconfig.get_config_var("SOABI") in native.CALLS_PATH.name


def test_the_module_is_built_where_it_is_stale_and_replaced_whole(tmp_path, monkeypatch):
    (tmp_path / "sglang_amd.h").write_text(HEADER)
    header, out = tmp_path / "sglang_amd.h", tmp_path / "_calls.so"
    if build.build_calls(out, header) is None:
        pytest.skip("no Python headers")
    first = out.stat()
    assert build.build_calls(out, header) == out and out.stat() == first                # nothing to do
    os.utime(header, (first.st_atime + 2, first.st_mtime + 2))
    with out.open("rb") as reader:                                                      # (holds the old file)
        monkeypatch.setenv("HIPCC", "/bin/false")
        with pytest.raises(RuntimeError):
            build.build_calls(out, header)
        assert out.stat() == first                                                      # a failure leaves the old one
        monkeypatch.delenv("HIPCC")
        build.build_calls(out, header)
        assert out.stat().st_ino != first.st_ino and os.fstat(reader.fileno()).st_ino == first.st_ino
    made = out.stat()
    build.build_calls(out, header, force=True)
    assert out.stat().st_ino != made.st_ino and sorted(p.name for p in tmp_path.iterdir()) == ["_calls.so", "sglang_amd.h"]
