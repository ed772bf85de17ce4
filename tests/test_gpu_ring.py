"""The int8 row-scale product on 128 x 128 tiles with the eight-stage LDS ring (at most one workgroup per
compute unit, K in whole rounds of the ring) and with the four-stage one beside it: outputs against the
exact int32 sums, bit for bit in fp32."""
import numpy as np
import pytest
import torch

from kitchen_amd import ops
from oracle import gemm

pytestmark = pytest.mark.gpu


# K groups: one round of eight, one with a dead group, an odd number of blocks of four (four stages),
# two rounds, many; split along K (K = 12288, K = 8192); ragged M and N; a full grid and past it
@pytest.mark.parametrize("m,n,k", [(129, 17, 512), (256, 300, 448), (200, 260, 768), (300, 2000, 960), (256, 640, 12288),
                                   (130, 128, 8192), (1024, 3072, 512), (640, 6500, 1024), (2048, 2050, 512)])
@pytest.mark.parametrize("tiled", [False, True])
def test_row_scale(gpu_device, m, n, k, tiled):
    print(f"[ring] M={m} N={n} K={k} tiled={tiled}", flush=True)
    rng = np.random.default_rng(m + n + k)
    qa = rng.integers(-127, 128, (m, k)).astype(np.int8)
    qw = rng.integers(-127, 128, (n, k)).astype(np.int8)
    sa, sw = rng.uniform(0.01, 0.02, m).astype(np.float32), rng.uniform(0.001, 0.002, n).astype(np.float32)
    bias = rng.standard_normal(n).astype(np.float32)
    d = lambda a: torch.from_numpy(a).to(gpu_device)                      # noqa: E731
    w = ops.tile_int8_weight(d(qw)) if tiled else d(qw)
    y = ops.gemm_rowscale(d(qa), d(sa), w, d(sw), d(bias), n, 8, out_dtype=torch.float32)
    torch.cuda.synchronize()
    rows = np.r_[0:min(m, 140), max(0, m - 140):m]
    p = gemm.partials(qa[rows], qw, k)[0].astype(np.float32)
    assert np.array_equal(y.cpu().numpy()[rows], (p * sa[rows, None]) * sw + bias)
