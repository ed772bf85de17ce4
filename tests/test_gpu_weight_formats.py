"""The offline weight quantizer and the codebook decoder at the edges of their layouts (csrc/mq_wquant.hip:
1024-column chunks, four waves per row in the row formats; csrc/mq_codebook.hip: 16-row tiles), against
the oracle, byte for byte."""
import numpy as np
import pytest
import torch

import kitchen_amd as ck
from kitchen_amd import _lib, ops, weights
from oracle import codebook as cbk
from oracle import linear, quant

pytestmark = pytest.mark.gpu


def _rot(w, cg):
    return linear.rotate_weight(w, cg) if cg else w


# K: one group, groups odd in number, a chunk's end, one past it, four chunks, past four and sixteen
# (2, 4 and 8 chunks per wave of the row formats); N: a lone row, a ragged last workgroup
@pytest.mark.parametrize("n,k,cg", [(1, 64, 64), (3, 192, 16), (5, 1024, 256), (7, 1088, 64), (2, 4096, 256),
                                    (3, 4352, 256), (2, 8256, 64), (1, 16448, 16), (2, 320, 0)])
@pytest.mark.parametrize("shift", [0, 1])
def test_quantizers(gpu_device, n, k, cg, shift):
    """shift: the weight starts one element into an odd-strided buffer (element-wise loads)."""
    print(f"[wquant] N={n} K={k} cg={cg} shift={shift}", flush=True)
    rng = np.random.default_rng(n * k + cg)
    w = (rng.standard_normal((n, k)) * 0.02).astype(np.float32)
    w[:, 5::61] *= 30.0
    if n > 1:
        w[1, :64] = 0.0
    for dtype in (torch.bfloat16, torch.float32):
        buf = torch.zeros((n, k + 3 * shift), dtype=dtype, device=gpu_device)
        t = buf[:, shift:shift + k]
        t.copy_(torch.from_numpy(w).to(dtype))
        r = _rot(t.float().cpu().numpy(), cg)
        q, s, z = weights.quantize_w4a8_asym_weight(t, 64, cg)
        q0, s0, z0 = quant.quant_weight_u4_asym(r, 64)
        assert np.array_equal(q.cpu().numpy(), quant.pack_u4(q0)) and np.array_equal(z.cpu().numpy(), quant.pack_u4(z0))
        assert np.array_equal(s.cpu().numpy().view(np.uint16), s0.view(np.uint16))
        q, s = weights.quantize_w4a4_group_weight(t, 64, cg)
        q0, s0 = quant.quant_weight_i4_sym_group(r, 64)
        assert np.array_equal(q.cpu().numpy(), quant.pack_i4(q0))
        assert np.array_equal(s.cpu().numpy().view(np.uint16), s0.view(np.uint16))
        q, s = weights.quantize_int8_convrot_weight(t, cg or None)
        q0, s0 = quant.quant_weight_i8_rowwise(r)
        assert np.array_equal(q.cpu().numpy(), q0) and np.array_equal(s.cpu().numpy().view(np.uint32), s0.view(np.uint32))
        if cg:
            q, s = weights.quantize_convrot_w4a4_weight(t, cg, 64)
            q0, s0 = quant.quant_weight_i4_rowwise(r)
            assert np.array_equal(q.cpu().numpy(), quant.pack_i4(q0))
            assert np.array_equal(s.cpu().numpy().view(np.uint32), s0.view(np.uint32))


def test_ties_and_small_scales(gpu_device):
    """Weights on half-integer multiples of their scale, and groups whose fp16 scale is subnormal."""
    print("[wquant] ties, subnormal scales", flush=True)
    rng = np.random.default_rng(5)
    w = rng.integers(-15, 16, (8, 256)).astype(np.float32) * 0.5
    w[:, ::64] = 7.0                                  # int4 scale exactly 1 (and 127: int8 ties below)
    w[4:] *= np.float32(2.0 ** -26)                   # fp16 scales 2^-24 k or 0
    t = torch.from_numpy(w).to(gpu_device)
    for fn, ref in ((weights.quantize_w4a4_group_weight, quant.quant_weight_i4_sym_group),
                    (weights.quantize_w4a8_asym_weight, quant.quant_weight_u4_asym)):
        got, want = fn(t, 64, 0), ref(w, 64)
        pack = quant.pack_i4 if fn is weights.quantize_w4a4_group_weight else quant.pack_u4
        assert np.array_equal(got[0].cpu().numpy(), pack(want[0]))
        assert np.array_equal(got[1].cpu().numpy().view(np.uint16), want[1].view(np.uint16))
    w8 = rng.integers(-253, 254, (4, 256)).astype(np.float32) * 0.5
    w8[:, 0] = 127.0
    q, s = weights.quantize_int8_convrot_weight(torch.from_numpy(w8).to(gpu_device), None)
    q0, s0 = quant.quant_weight_i8_rowwise(w8)
    assert np.array_equal(q.cpu().numpy(), q0) and np.array_equal(s.cpu().numpy(), s0)


def test_nan_and_infinite_weights(gpu_device):
    """NaN weights are left out of the extremes and get the clamp's lower bound; an infinite weight makes a
    row scale infinite and every finite code 0."""
    print("[wquant] NaN, inf", flush=True)
    w = torch.linspace(-1.0, 1.0, 256, device=gpu_device).repeat(4, 1)
    clean = weights.quantize_w4a4_group_weight(w, 64, 0)
    w[0, 5], w[1, 70] = float("nan"), float("nan")
    q, s = weights.quantize_w4a4_group_weight(w, 64, 0)
    q = q.view(torch.uint8)
    assert torch.equal(s, clean[1]) and (int(q[0, 2]) >> 4) == 9 and (int(q[1, 35]) & 15) == 9     # -7
    q, s, _ = weights.quantize_w4a8_asym_weight(w, 64, 0)
    assert torch.isfinite(s).all() and (int(q[0, 2]) >> 4) == 0 and (int(q[1, 35]) & 15) == 0
    w[2, 9] = float("inf")
    q, s = weights.quantize_int8_convrot_weight(w, None)
    assert int(q[0, 5]) == -127 and torch.isfinite(s[0]) and torch.isinf(s[2])
    assert int(q[2, 9]) == -127 and int(q[2].abs().sum()) == 127


def test_overflow_is_reported_once_per_call(gpu_device):
    w = torch.full((4, 2048), 1.0, device=gpu_device)
    w[3, 2000:] = 3.0e6
    with pytest.raises(ValueError, match="overflows the fp16 scale"):
        weights.quantize_w4a4_group_weight(w, 64, 0)
    weights.quantize_w4a4_group_weight(w[:3], 64, 0)      # the flag is the call's own


@pytest.mark.parametrize("n,k,gs", [(1, 192, 4), (16, 256, 8), (17, 1024, 16), (40, 1088, 32), (33, 3072, 64), (5, 192, 192)])
@pytest.mark.parametrize("shift", [0, 4])
def test_decode_to_tiles(gpu_device, n, k, gs, shift):
    """PreparedW4A8's tiles: the decoded rows, tiled; shift: packed rows aligned to 4 bytes only."""
    print(f"[codebook] tiles N={n} K={k} gs={gs} shift={shift}", flush=True)
    rng = np.random.default_rng(n + k + gs)
    qd = rng.integers(0, 256, (n, k // 2), dtype=np.uint8)
    sr = rng.integers(0, 256, (n, k // gs), dtype=np.uint8)            # every fp8 byte, NaN included
    sc = rng.uniform(0.001, 0.05, n).astype(np.float32)
    cb = np.sort(rng.uniform(-1, 1, 16)).astype(np.float32)
    buf = torch.zeros((n, k // 2 + shift), dtype=torch.uint8, device=gpu_device)
    q = buf[:, shift:] if shift else buf
    q.copy_(torch.from_numpy(qd))
    q0, _ = cbk.decode_w4a8_codebook(qd, sr, sc, cb, gs)
    args = (torch.from_numpy(sr).to(gpu_device), torch.from_numpy(sc).to(gpu_device), torch.from_numpy(cb).to(gpu_device))
    rows, rs = torch.empty((n, k), dtype=torch.int8, device=gpu_device), torch.empty(n, device=gpu_device)
    tiles = torch.full(((n + 15) // 16, k // 64, 16, 64), 99, dtype=torch.int8, device=gpu_device)
    head = (q.data_ptr(), q.stride(0), args[0].data_ptr(), k // gs, args[1].data_ptr(), args[2].data_ptr(), gs, n, k)
    _lib.call("mq_decode_w4a8_codebook", *head, rows.data_ptr(), k, rs.data_ptr(), _lib.stream_of(q))
    assert np.array_equal(rows.cpu().numpy(), q0) and np.array_equal(rs.cpu().numpy(), sc)
    rs.zero_()
    _lib.call("mq_decode_w4a8_codebook_tile16", *head, tiles.data_ptr(), rs.data_ptr(), _lib.stream_of(q))
    assert torch.equal(tiles, ops.tile_int8_weight(rows)) and np.array_equal(rs.cpu().numpy(), sc)
    p = ck.PreparedW4A8(q, *args, gs)
    assert (p.n, p.k) == (n, k) and torch.equal(p.q8, tiles) and torch.equal(p.row_scale, rs)


@pytest.mark.parametrize("cg", [0, 64, 256])
def test_nan_in_groups_of_scale_zero(gpu_device, cg):
    """A group whose scale is 0 (wholly NaN, as one NaN weight makes its whole Hadamard block, or too
    small for fp16) stores codes and zero-points of 0, NaN weights included."""
    print(f"[wquant] NaN, scale 0, cg={cg}", flush=True)
    w = torch.linspace(-1.0, 1.0, 512, device=gpu_device).repeat(3, 1)
    w[0, 64:128] = float("nan")
    w[1, 300] = float("nan")
    w[2, :256] = 1.0e-9
    w[2, 7] = float("nan")
    for fn in (weights.quantize_w4a4_group_weight, weights.quantize_w4a8_asym_weight):
        out = fn(w, 64, cg)
        q, s = out[0].view(torch.uint8).view(3, 8, 32).cpu(), out[1].float().cpu()
        zero = s == 0
        assert zero[0, 1] and zero[2, 0] and (cg == 0 or zero[1].any())
        assert not q[zero].any() and q[~zero].any()
        if len(out) == 3:
            z = torch.stack([out[2].cpu() & 15, out[2].cpu() >> 4], 2).view(3, 8)
            assert not z[zero].any()


def test_group_formats_under_a_default_device(gpu_device):
    """With a default device set, as loaders that build modules on the GPU do: the overflow flag is host
    memory whatever the default is."""
    print("[wquant] default device", flush=True)
    w = torch.linspace(-1.0, 1.0, 512, device=gpu_device).repeat(3, 1)
    want = weights.quantize_w4a8_asym_weight(w, 64, 64) + weights.quantize_w4a4_group_weight(w, 64, 64)
    with torch.device(gpu_device):
        got = weights.quantize_w4a8_asym_weight(w, 64, 64) + weights.quantize_w4a4_group_weight(w, 64, 64)
        with pytest.raises(ValueError, match="overflows the fp16 scale"):
            weights.quantize_w4a4_group_weight(w * 1e7, 64, 64)
    assert all(torch.equal(a, b) for a, b in zip(got, want))


@pytest.mark.parametrize("n,k,gs", [(17, 960, 48), (5, 1280, 80), (3, 2016, 112), (16, 1024, 1024), (33, 3072, 768)])
def test_decode_group_sizes(gpu_device, n, k, gs):
    """Groups that are no power of two, and one group a row: rows and, where K allows, tiles."""
    print(f"[codebook] group sizes N={n} K={k} gs={gs}", flush=True)
    rng = np.random.default_rng(gs)
    qd = rng.integers(0, 256, (n, k // 2), dtype=np.uint8)
    sr, sc = rng.integers(0, 256, (n, k // gs), dtype=np.uint8), rng.uniform(0.001, 0.05, n).astype(np.float32)
    cb = np.sort(rng.uniform(-1, 1, 16)).astype(np.float32)
    q0, _ = cbk.decode_w4a8_codebook(qd, sr, sc, cb, gs)
    args = [torch.from_numpy(a).to(gpu_device) for a in (qd, sr, sc, cb)]
    q, _ = ops.decode_w4a8_codebook_weight(*args, gs)
    assert np.array_equal(q.cpu().numpy(), q0)
    if k % 64 == 0:
        assert torch.equal(ck.PreparedW4A8(*args, gs).q8, ops.tile_int8_weight(q))
