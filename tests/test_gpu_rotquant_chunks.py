"""Rotate + quantize at the chunk counts that leave a wave's last 1024-column chunk past the row's end, one
group above and below each such edge: row-major codes against the oracle, codes in 16-row tiles through the
W8A8 linear against the same linear on row-major codes, bit for bit."""
import numpy as np
import pytest
import torch

from kitchen_amd import _lib, ops, synth
from oracle import quant, swiglu
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


@pytest.mark.parametrize("k", [5120, 9216, 14336])
@pytest.mark.parametrize("mode", [_lib.SWIGLU_FUSED, _lib.SWIGLU_EAGER])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_dead_chunk_swiglu(gpu_device, k, mode, dtype):
    """SwiGLU rows whose waves leave a last chunk, more of them than workgroups are resident (3 on each of
    256 compute units, one or two rows a step), with gates outside the silu table (0, 200 and -200) in some lanes,
    whole chunks and whole rows."""
    m = 2100
    print(f"[chunks] swiglu M={m} K={k} eager={mode == _lib.SWIGLU_EAGER} {dtype}", flush=True)
    rng = np.random.default_rng(k)
    g, u = (rng.standard_normal((m, k)).astype(np.float32) * 3 for _ in range(2))
    g[rng.random((m, k)) < 0.0005] = 0.0
    g[::7, 17], g[::5, 1024:2048], g[3::11, -1] = 200.0, -200.0, 200.0
    g[5::13] = 0.0
    h = torch.from_numpy(np.concatenate([g, u], axis=1)).to(dtype).to(gpu_device)
    rows = np.r_[0:120, m // 2:m // 2 + 60, m - 60:m]
    q0, s0 = swiglu.swiglu_rotquant(h[rows].float().cpu().numpy(), 256, 4, dtype="f16" if dtype == torch.float16 else "bf16",
                                    eager=mode == _lib.SWIGLU_EAGER)
    q, s = ops.rotate_quantize(h, 256, 4, True, swiglu=mode)
    assert np.array_equal(s[rows].cpu().numpy().view(np.uint32), s0.view(np.uint32))
    assert np.array_equal(q[rows].cpu().numpy(), quant.pack_i4(q0))


@pytest.mark.parametrize("k", [5120, 9216, 14336])
def test_dead_chunk_other_inputs(gpu_device, k):
    """fp32 input, and the x16 code layout, at rows whose waves leave a last chunk."""
    m = 1100
    print(f"[chunks] fp32, x16alt M={m} K={k}", flush=True)
    xb = synth.activations(m, k, seed=k)
    _check(xb[:40], 256, 4, _lib.Q_X16ALT, gpu_device, "chunks")
    x = synth.bf16_bits_to_f32(xb) * np.float32(1.0 + 2.0 ** -12)   # fp32 values between the bf16 ones
    q, s = ops.rotate_quantize(torch.from_numpy(x).to(gpu_device), 256, 8)
    rows = np.r_[0:30, m - 30:m]
    q0, s0 = quant.rotquant(x[rows], 256, 8)
    assert np.array_equal(s[rows].cpu().numpy().view(np.uint32), s0.view(np.uint32))
    assert np.array_equal(q[rows].cpu().numpy(), q0)
