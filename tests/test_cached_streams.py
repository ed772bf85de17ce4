"""Weights that the linears expand or decode once and keep: a call on another stream than the one that made them
waits for them, and keeps them from being reused while it runs. On the CPU, with stand-ins for the streams;
on the GPU, with a first call still queued behind other work when a second stream's call is made."""
import types

import pytest
import torch

from kitchen_amd import _lib, ops


class _Buffer:
    def __init__(self):
        self.recorded = []

    def record_stream(self, stream):
        self.recorded.append(stream)


@pytest.fixture
def streams(monkeypatch):
    """Streams 1 and 2: state["now"] is the current one, state["waits"] the streams that waited for the device."""
    state = {"now": 1, "capturing": False, "waits": []}
    monkeypatch.setattr(torch.cuda, "synchronize", lambda device=None: state["waits"].append(state["now"]))
    monkeypatch.setattr(torch.cuda, "current_stream", lambda device=None: state["now"])
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: state["capturing"])
    monkeypatch.setattr(_lib, "stream_of_device", lambda device: state["now"])
    return state


def _check(state, call, buffers):
    made = call()
    assert call() is made and not any(b.recorded for b in buffers)
    state["now"], state["capturing"] = 2, True   # a capture neither waits nor counts as the stream's first use
    assert call() is made and not state["waits"]
    state["capturing"] = False
    assert call() is made and call() is made
    assert state["waits"] == [2] and all(b.recorded == [2] for b in buffers)
    state["now"] = 1
    assert call() is made and state["waits"] == [2]


@pytest.mark.parametrize("layout,m", [(_lib.ACT_I8, 200), (_lib.W4X_ROW, 5)])
def test_expansion_on_another_stream(streams, monkeypatch, layout, m):
    buf = _Buffer()
    monkeypatch.setattr(ops, "expand_w4_weight", lambda *a: types.SimpleNamespace(buf=buf))
    w, s = torch.zeros((32, 128), dtype=torch.uint8), torch.ones((32, 4), dtype=torch.float16)
    scales = None if layout == _lib.W4X_ROW else s
    _check(streams, lambda: ops._expansion(w, None, layout, m, 256, scales, streams["now"]), [buf])


def test_decoded_weight_on_another_stream(streams, monkeypatch):
    dec = (_Buffer(), _Buffer())
    monkeypatch.setattr(ops, "decode_w4a8_codebook_weight", lambda *a: dec)
    q, t = torch.zeros((32, 128), dtype=torch.int8), torch.ones(32)
    _check(streams, lambda: ops._decoded_w4a8(q, t, t, None, 16), dec)


@pytest.mark.gpu
@pytest.mark.parametrize("fmt", ["group", "row", "codebook"])
def test_second_stream_uses_a_weight_that_is_being_made(gpu_device, fmt):
    print(f"[streams] {fmt}", flush=True)
    n, k, m = 6144, 4096, 256
    gen = torch.Generator(device=gpu_device).manual_seed(1)
    q = torch.randint(-128, 128, (n, k // 2), generator=gen, device=gpu_device, dtype=torch.int8)
    s16 = (torch.rand(n, k // 64, generator=gen, device=gpu_device) * 0.01).half()
    s = torch.rand(n, generator=gen, device=gpu_device) * 0.01
    s8 = (torch.rand(n, k // 16, generator=gen, device=gpu_device) * 40).to(torch.float8_e4m3fn)
    x = torch.randn(m, k, generator=gen, device=gpu_device).bfloat16()

    def linear(weight):
        if fmt == "codebook":
            return ops.w4a8_int8_linear(x, weight, s8, s, None, None, None, 16, 256, torch.bfloat16)
        return ops.convrot_w4a4_linear(x, weight, s16 if fmt == "group" else s, None, 256)

    want = linear(q.clone())
    a, b = torch.cuda.Stream(), torch.cuda.Stream()
    work = torch.randn(4096, 4096, generator=gen, device=gpu_device)
    weight = q.clone()
    torch.cuda.synchronize()
    with torch.cuda.stream(a):
        for _ in range(20):
            work = work @ work * 1e-4
        first = linear(weight)
    with torch.cuda.stream(b):
        second = linear(weight)
    torch.cuda.synchronize()
    assert torch.equal(first, want) and torch.equal(second, want)
