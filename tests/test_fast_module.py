"""The CPython module of the per-call entry points (_fast.so): which arguments may be missing, whether a module
built from another header is noticed, and the ctypes calls that take its place where it is not built. CPU
only: every call is refused or empty, so nothing is launched."""
import ctypes
import os
import subprocess
import sys

import pytest

from conftest import PKG_ROOT
from kitchen_amd import _lib
from test_fast_calls import CASES

POINTERS = {name: [i for i, t in enumerate(_lib._SIGNATURES[name][0]) if t is ctypes.c_void_p] for name in _lib.FAST_ENTRIES}


@pytest.mark.parametrize("name,args,rows,bad", CASES, ids=[c[0] for c in CASES])
def test_none_is_a_null_pointer_and_nothing_else(name, args, rows, bad):
    """As through ctypes: a missing pointer may be None, a missing size or option is refused (taken as 0 it
    would be a silent no-op, or no rotation)."""
    lib = _lib.load()
    empty = list(args)
    empty[rows] = 0
    for i in range(len(args)):
        one = empty[:i] + [None] + empty[i + 1:]
        if i in POINTERS[name]:
            assert _lib._entries[name](*one) == getattr(lib, name)(*one)
        else:
            with pytest.raises(ctypes.ArgumentError):
                getattr(lib, name)(*one)
            with pytest.raises(TypeError, match=f"argument {i + 1} "):
                _lib._entries[name](*one)


def _python(code):
    env = dict(os.environ, PYTHONPATH=PKG_ROOT)
    return subprocess.run([sys.executable, "-c", code], capture_output=True, text=True, env=env, timeout=300)


def test_a_module_of_another_abi_version_is_refused():
    """The order of an entry's arguments is compiled into the module: one built from an older header is not bound."""
    res = _python("""
import sys, types
from kitchen_amd import _lib
stale = types.ModuleType("kitchen_amd._fast")
stale.ABI_VERSION = _lib.ABI_VERSION - 1
stale.bind = lambda *a: print("bound")
for name in _lib.FAST_ENTRIES:
    setattr(stale, name, lambda *a: 0)
sys.modules["kitchen_amd._fast"] = stale
import kitchen_amd
kitchen_amd._fast = stale
try:
    _lib.load()
except RuntimeError as e:
    print("refused:", e)
""")
    assert res.returncode == 0, res.stderr
    assert "bound" not in res.stdout and "refused: " in res.stdout and "rebuild" in res.stdout


def test_without_the_module_the_calls_go_through_ctypes():
    """Where _fast.so is not built, the same library's entries are called through ctypes, with a warning."""
    res = _python("""
import sys, warnings
sys.modules["kitchen_amd._fast"] = None
from kitchen_amd import _lib
with warnings.catch_warnings(record=True) as seen:
    warnings.simplefilter("always")
    lib = _lib.load()
assert len(seen) == 1 and "_fast.so" in str(seen[0].message), seen
for name in _lib.FAST_ENTRIES:
    assert _lib._entries[name] is getattr(lib, name)
A = 1 << 20
_lib.call("mq_rotquant", A, 0, 0, 256, 256, 256, 8, 0, A, 256, A, None)
try:
    _lib.call("mq_rotquant", A, 0, 4, 256, 256, 256, 5, 0, A, 256, A, None)
except ValueError as e:
    print("refused:", e)
""")
    assert res.returncode == 0, res.stderr
    assert "refused: mq_rotquant" in res.stdout


@pytest.mark.parametrize("missing", ["headers", "compiler"])
def test_build_without_headers_or_compiler(monkeypatch, tmp_path, missing):
    """The library is built all the same, and no module of an earlier build is left behind."""
    import build

    fast = tmp_path / "_fast.so"
    fast.write_bytes(b"old")
    monkeypatch.setattr(build, "FAST", str(fast))
    if missing == "headers":
        monkeypatch.setattr(build.sysconfig, "get_paths", lambda: {"include": str(tmp_path)})
    else:
        monkeypatch.setattr(build, "hipcc", lambda: str(tmp_path / "hipcc"))
        monkeypatch.setattr(build.shutil, "which", lambda name: None)
    build._compile_fast()
    assert not fast.exists()
