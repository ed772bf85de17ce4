"""The host side of the linears, on the CPU: what is handed to the library, what comes back, and the
workspaces that calls share. The library is called with no rows, so nothing is launched."""
import gc
import threading
import weakref

import pytest
import torch

from kitchen_amd import _lib, ops

ROWS = {"mq_linear_w4_group": 17, "mq_linear_rowscale": 15}   # index of the argument that counts the rows


@pytest.fixture
def calls(monkeypatch):
    """Host tensors in place of device tensors: each call's arguments are kept, and handed to the library
    itself with a row count of 0."""
    _lib.load()
    seen = []

    def call(name, *args):
        seen.append((name, args))
        empty = list(args)
        empty[ROWS[name]] = 0
        assert _lib._entries[name](*empty) == 0

    monkeypatch.setattr(ops, "_as_2d", lambda x, k: x.reshape(-1, k))
    monkeypatch.setattr(ops, "_linear_workspace", lambda *a: torch.empty(256, dtype=torch.uint8))
    monkeypatch.setattr(_lib, "stream_of_device", lambda device: 0)
    monkeypatch.setattr(_lib, "call", call)
    return seen


def _linears(x, cg):
    """One linear of each library entry point, N = 8, K = 256."""
    n, k = 8, 256
    q, s16 = torch.zeros((n, k // 2), dtype=torch.uint8), torch.ones((n, k // 64), dtype=torch.float16)
    return [ops.w4a8_int8_linear(x, q, s16, None, None, None, None, 64, cg, x.dtype),
            ops.convrot_w4a4_linear(x, q.view(torch.int8), s16, None, cg),
            ops.convrot_w4a4_linear(x, q.view(torch.int8), torch.ones(n), None, cg),
            ops.int8_linear(x, torch.zeros((n, k), dtype=torch.int8), torch.ones((n, 1)), None, x.dtype, True, cg)]


@pytest.mark.parametrize("cg", [256, 256.0, torch.tensor(256)])
def test_convrot_groupsize_of_any_number_type(calls, cg):
    """Whatever int() takes: a checkpoint's metadata may hold the group size as a float."""
    ys = _linears(torch.zeros((3, 256), dtype=torch.bfloat16), cg)
    assert [y.shape for y in ys] == [(3, 8)] * 4 and len(calls) == 4
    assert all(args[3] == 256 for _, args in calls)


def test_outputs_are_plain_tensors(calls):
    """The outputs are the library's own buffers, not the class of the activations."""
    class Tagged(torch.Tensor):
        pass

    for dtype in (torch.bfloat16, torch.float32):
        x = torch.zeros((3, 256), dtype=dtype)
        assert [type(y) for y in _linears(x.as_subclass(Tagged), 256)] == [torch.Tensor] * 4
        assert [(type(y), y.dtype, y.device) for y in _linears(x, 256)] == [(torch.Tensor, dtype, x.device)] * 4


def test_threads_on_one_stream_have_their_own_workspaces(monkeypatch):
    """A linear launches twice (codes into the workspace, then the product that reads them) and its call
    releases the GIL: a second thread on the same stream may not be handed the same workspace."""
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: False)
    cpu, got, refs = torch.device("cpu"), {}, {}
    barrier = threading.Barrier(2)

    def work(name):
        a = ops._scratch(1000, cpu, 7)
        barrier.wait(10)
        got[name] = (a.data_ptr(), ops._scratch(900, cpu, 7) is a, ops._scratch(1000, cpu, 8) is a)
        refs[name] = weakref.ref(a)
        barrier.wait(10)

    threads = [threading.Thread(target=work, args=(i,)) for i in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join(20)
    assert got[0][0] != got[1][0]
    assert all(again and not other for _, again, other in got.values())   # kept per stream, in each thread
    gc.collect()
    assert refs[0]() is None and refs[1]() is None                        # and given back when it ends
