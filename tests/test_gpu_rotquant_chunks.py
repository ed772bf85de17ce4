"""Rotate + quantize at the chunk counts that leave a wave's last 1024-column chunk past the row's end, one
group above and below each such edge: row-major codes against the oracle, codes in 16-row tiles through the
W8A8 linear against the same linear on row-major codes, bit for bit."""
import pytest
import torch

from kitchen_amd import _lib, ops, synth
from test_gpu_rotquant import _check

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m,k", [(3, 2048), (37, 3328), (5, 5120), (5, 7168), (1027, 5120), (1027, 5376), (1027, 7168),
                                 (1027, 7424), (19, 9216), (19, 11264), (19, 11520), (19, 13312), (19, 15360),
                                 (19, 15616)])
def test_dead_chunk_codes(gpu_device, m, k):
    xb = synth.activations(m, k, seed=m + k)
    _check(xb, 256, 8, False, gpu_device, "chunks")
    _check(xb, 64, 4, True, gpu_device, "chunks")


@pytest.mark.parametrize("m,k", [(129, 2048), (1027, 5120), (1027, 5376), (300, 9216), (300, 11520), (300, 14336)])
def test_dead_chunk_tiles(gpu_device, m, k):
    n = 256
    print(f"[chunks] w8a8 tiles M={m} K={k}", flush=True)
    x = synth.to_bf16_tensor(synth.activations(m, k, seed=k), gpu_device)
    gen = torch.Generator(device=gpu_device).manual_seed(k)
    w = torch.randint(-127, 128, (n, k), generator=gen, device=gpu_device, dtype=torch.int8)
    s = torch.rand(n, generator=gen, device=gpu_device) * 2e-4 + 3e-4
    bias = torch.zeros(n, dtype=torch.bfloat16, device=gpu_device)
    qa, sa = ops.rotate_quantize(x, 256, 8, _lib.Q_BYTES)
    y2 = ops.gemm_rowscale(qa, sa, w, s, bias, n, 8)
    y1 = ops.int8_linear(x, w, s, bias, torch.bfloat16, True, 256)
    torch.cuda.synchronize()
    assert torch.equal(y1.view(torch.int16), y2.view(torch.int16))
