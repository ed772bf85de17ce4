"""The CPython calls of the per-call entry points (csrc/mq_fast.c): the library's own status and messages, as
through ctypes, and refusals of a wrong argument list. CPU only: every call fails validation or is
empty, so nothing is launched."""
import pytest

from kitchen_amd import _lib

A = 1 << 20   # a fake aligned address: never dereferenced

# (entry, arguments, index of the argument that counts the rows, a bad value for one argument)
CASES = [
    ("mq_rotquant", [A, 0, 4, 256, 256, 256, 8, 0, A, 256, A, None], 2, (6, 5)),
    ("mq_swiglu_rotquant", [A, 0, 4, 256, 512, 256, 8, 0, 1, A, 256, A, None], 2, (8, 7)),
    ("mq_linear_w4_group", [A, 0, 256, 256, 8, 0, A, 128, A, 4, A, 2, None, 0, A, 0, 64, 4, 64, 256, A, 1 << 20, None],
     17, (4, 5)),
    ("mq_linear_rowscale", [A, 0, 256, 256, 8, 0, A, 256, 8, A, None, 0, A, 0, 64, 4, 64, 256, A, 1 << 20, None], 15,
     (8, 5)),
]


@pytest.mark.parametrize("name,args,rows,bad", CASES, ids=[c[0] for c in CASES])
def test_same_status_and_message(name, args, rows, bad):
    lib = _lib.load()
    fast, slow = _lib._entries[name], getattr(lib, name)
    assert fast is not slow and name in _lib.FAST_ENTRIES
    empty = list(args)
    empty[rows] = 0
    assert fast(*empty) == slow(*empty) == 0
    wrong = list(args)
    wrong[bad[0]] = bad[1]
    assert slow(*wrong) == -1
    message = lib.mq_last_error()
    assert fast(*wrong) == -1 and lib.mq_last_error() == message != b""
    with pytest.raises(ValueError, match=name):
        _lib.call(name, *wrong)


@pytest.mark.parametrize("name,args,rows,bad", CASES, ids=[c[0] for c in CASES])
def test_argument_list(name, args, rows, bad):
    _lib.load()
    with pytest.raises(TypeError, match="arguments"):
        _lib._entries[name](*args[:-1])
    with pytest.raises(TypeError):
        _lib._entries[name](*args[:-1], "stream")
    with pytest.raises(OverflowError):
        _lib._entries[name](1 << 70, *args[1:])
