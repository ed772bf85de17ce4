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
