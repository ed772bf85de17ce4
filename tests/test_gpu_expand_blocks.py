"""mq_expand_weight_w4 where its launches split: scale pairs over more than one block of 256 (N > 8k), group
counts around multiples of four, a last band of one row, tiles around a multiple of a workgroup's four waves.
The bytes are compared with the restatement of the layout that test_gpu_expand checks against."""
import numpy as np
import pytest
import torch

import kitchen_amd as ck
from kitchen_amd import _lib
from test_gpu_expand import _expand_np, _scale_pairs_np

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("layout,asym", [(_lib.ACT_I8, True), (_lib.ACT_X16ALT, True), (_lib.ACT_X16ALT, False),
                                         (_lib.W4X_ROW, False)])
@pytest.mark.parametrize("n,k", [(7905, 256), (8193, 320), (8209, 64), (1, 16448), (17, 448)])
def test_expansion_blocks(gpu_device, layout, asym, n, k):
    print(f"[expand] blocks n={n} k={k} asym={asym} layout={layout}", flush=True)
    rng = np.random.default_rng(n + k)
    qw = rng.integers(0, 256, (n, k // 2), dtype=np.uint8)
    wz = rng.integers(0, 256, (n, (k // 64 + 1) // 2), dtype=np.uint8) if asym else None
    s16 = rng.integers(0, 0x7c00, (n, k // 64), dtype=np.uint16).view(np.float16)
    ex = ck.expand_w4_weight(torch.from_numpy(qw).to(gpu_device),
                             None if wz is None else torch.from_numpy(wz).to(gpu_device), layout,
                             None if layout == _lib.W4X_ROW else torch.from_numpy(s16).to(gpu_device))
    torch.cuda.synchronize()
    assert np.array_equal(ex.tiles.cpu().numpy(), _expand_np(qw, wz, n, k, layout))
    if layout != _lib.W4X_ROW:
        pairs = ex.buf[(n + 15) // 16 * 16 * k:].cpu().numpy().view(np.uint32)
        assert np.array_equal(pairs, _scale_pairs_np(s16, n, k).reshape(-1))
