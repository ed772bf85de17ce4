"""GPU parity of the few-row GEMM (5 <= M <= 128, csrc/mq_gemm_few.hip) at the edges of its blocks: rows
(16 per block), columns (16, 32 or 64 per workgroup), an odd number of K groups, fewer spans of K than
waves, unpaired scale rows, and both activation layouts (the whole linears' 16-row tiles, rows)."""
import numpy as np
import pytest
import torch

from kitchen_amd import _lib, ops, synth
from oracle import gemm, quant

pytestmark = pytest.mark.gpu

# (M, N, K): one and two row blocks, the last of every block count, N inside / at / past a block and on
# each workgroup width (N > 4096, N > 8192), one group, odd groups, spans not a multiple of the waves
SHAPES = [(5, 1, 64), (16, 17, 128), (17, 4096, 192), (33, 300, 1088), (48, 8200, 320), (65, 8193, 192),
          (80, 4100, 1024), (81, 513, 576), (96, 100, 3072), (113, 31, 448), (128, 4097, 640)]


def _t(a, dev):
    return torch.from_numpy(np.ascontiguousarray(a)).to(dev)


@pytest.mark.parametrize("m,n,k", SHAPES)
@pytest.mark.parametrize("kind", ["u4", "i4", "i4x16"])
def test_group_scale(gpu_device, m, n, k, kind):
    print(f"[few] group {kind} M={m} N={n} K={k}", flush=True)
    rng = np.random.default_rng(m * n + k)
    g = k // 64
    lim = 127 if kind == "u4" else 7
    qa = rng.integers(-lim, lim + 1, (m, k)).astype(np.int8)
    sa = rng.uniform(0.005, 0.015, m).astype(np.float32)
    s16 = rng.uniform(0.001, 0.01, (n, g)).astype(np.float16)
    bias = rng.standard_normal(n).astype(np.float32)
    if kind == "u4":
        q, z = rng.integers(0, 16, (n, k)).astype(np.uint8), rng.integers(0, 16, (n, g)).astype(np.uint8)
        w, wz, v = quant.pack_u4(q), _t(quant.pack_u4(z), gpu_device), gemm.zero_adjusted(q, z, 64)
    else:
        v = rng.integers(-8, 8, (n, k)).astype(np.int8)
        w, wz = quant.pack_i4(v), None
    codes, mode = qa, _lib.ACT_I8
    if kind == "i4x16":   # 16 * q, negated in odd groups
        sign = np.where(np.arange(k) // 64 % 2, -16, 16).astype(np.int8)
        codes, mode = (qa * sign).astype(np.int8), _lib.ACT_X16ALT
    y = ops.gemm_w4_group(_t(codes, gpu_device), _t(sa, gpu_device), _t(w, gpu_device), _t(s16, gpu_device), wz,
                          _t(bias, gpu_device), n, act_mode=mode, out_dtype=torch.float32)
    torch.cuda.synchronize()
    p = gemm.partials(qa, v, 64).astype(np.float64)                       # [G, M, N]
    terms = p * s16.T.astype(np.float64)[:, None, :]
    y0 = terms.sum(0) * sa[:, None] + bias
    # G fmas and at most 8 sums of waves, then the row scale and the bias: each rounds once
    bound = ((g + 8 + 2) * 2.0 ** -24) * (np.abs(terms).sum(0) * sa[:, None] + np.abs(bias)) + 1e-30
    assert (np.abs(y.cpu().numpy() - y0) <= bound).all()


@pytest.mark.parametrize("m,n,k", SHAPES)
@pytest.mark.parametrize("kind", ["i4", "i8", "tile"])
def test_row_scale(gpu_device, m, n, k, kind):
    if kind == "tile" and k < 192:
        pytest.skip("16-row tiles need K >= 192")
    print(f"[few] row {kind} M={m} N={n} K={k}", flush=True)
    rng = np.random.default_rng(m + n * k)
    qa = rng.integers(-127, 128, (m, k)).astype(np.int8)
    qw = rng.integers(-8, 8, (n, k)).astype(np.int8) if kind == "i4" else rng.integers(-127, 128, (n, k)).astype(np.int8)
    sa, sw = rng.uniform(0.01, 0.02, m).astype(np.float32), rng.uniform(0.001, 0.002, n).astype(np.float32)
    bias = rng.standard_normal(n).astype(np.float32)
    w = _t(quant.pack_i4(qw) if kind == "i4" else qw, gpu_device)
    if kind == "tile":
        w = ops.tile_int8_weight(w)
    y = ops.gemm_rowscale(_t(qa, gpu_device), _t(sa, gpu_device), w, _t(sw, gpu_device), _t(bias, gpu_device), n,
                          4 if kind == "i4" else 8, out_dtype=torch.float32)
    torch.cuda.synchronize()
    p = gemm.partials(qa, qw, k)[0].astype(np.float32)                    # exact int32 sums, converted
    assert np.array_equal(y.cpu().numpy(), (p * sa[:, None]) * sw + bias)


@pytest.mark.parametrize("m", [5, 16, 77, 128])
@pytest.mark.parametrize("n,k,pad", [(520, 1088, 0), (4100, 3072, 1), (48, 192, 1)])
def test_linears_read_tiles_as_rows(gpu_device, m, n, k, pad):
    """The whole linears' 16-row tiles of codes give the bits of the two-step path's rows; an odd scale
    stride (pad) takes the unpaired scale loads."""
    print(f"[few] linears M={m} N={n} K={k} pad={pad}", flush=True)
    x = synth.to_bf16_tensor(synth.activations(m, k, seed=m), gpu_device)
    rng = np.random.default_rng(k)
    qd = _t(rng.integers(0, 256, (n, k // 2)).astype(np.uint8), gpu_device)
    g = k // 64
    s16 = _t(rng.uniform(0.001, 0.01, (n, g + pad)).astype(np.float16), gpu_device)[:, :g]
    zp = _t(rng.integers(0, 256, (n, (g + 1) // 2)).astype(np.uint8), gpu_device)
    for bits, layout, mode in ((8, _lib.Q_BYTES, _lib.ACT_I8), (4, _lib.Q_X16ALT, _lib.ACT_X16ALT)):
        y1 = ops._linear_w4_group(x, False, 64, bits, qd, s16, zp, None, n, k, torch.bfloat16)
        qa, sa = ops.rotate_quantize(x, 64, bits, layout)
        y2 = ops.gemm_w4_group(qa, sa, qd, s16, zp, None, n, act_mode=mode)
        assert torch.equal(y1.view(torch.int16), y2.view(torch.int16))
    w8 = _t(rng.integers(-127, 128, (n, k)).astype(np.int8), gpu_device)
    sw = _t(rng.uniform(0.001, 0.002, n).astype(np.float32), gpu_device)
    y3 = ops.int8_linear(x, w8, sw, None, torch.bfloat16, True, 64)
    qa, sa = ops.rotate_quantize(x, 64, 8)
    y4 = ops.gemm_rowscale(qa, sa, ops.tile_int8_weight(w8), sw, None, n, 8)
    torch.cuda.synchronize()
    assert torch.equal(y3.view(torch.int16), y4.view(torch.int16))


@pytest.mark.parametrize("m,k", [(1, 32768 * 4 + 64), (2, 65536), (3, 43776), (4, 32832), (4, 65600)])
def test_rows_past_the_gemv(gpu_device, m, k):
    """One to four rows that the GEMV's LDS does not hold (M * K > 131072): the few-row kernel to K = 65536, the
    128 x 128-tile kernel past it."""
    n = 48
    print(f"[few] long rows M={m} K={k}", flush=True)
    rng = np.random.default_rng(m + k)
    qa = rng.integers(-127, 128, (m, k)).astype(np.int8)
    qw = rng.integers(-127, 128, (n, k)).astype(np.int8)
    sa, sw = rng.uniform(0.01, 0.02, m).astype(np.float32), rng.uniform(0.001, 0.002, n).astype(np.float32)
    y = ops.gemm_rowscale(_t(qa, gpu_device), _t(sa, gpu_device), _t(qw, gpu_device), _t(sw, gpu_device), None, n, 8,
                          out_dtype=torch.float32)
    torch.cuda.synchronize()
    p = gemm.partials(qa, qw, k)[0].astype(np.float32)
    assert np.array_equal(y.cpu().numpy(), (p * sa[:, None]) * sw)
