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
