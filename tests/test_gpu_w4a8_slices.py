"""W4A8 GEMMs of more than 64 tokens on narrow weights: slices of equal token tiles
side by side (65..512 tokens, at most two workgroups of 16 weight rows a CU), at the
edges of the slices and of the rule, ragged N, bias and strided activation rows; and
the tile kernel's one- and two-step K and its last rows beyond the rule.  Bit for bit
against the oracle."""
import numpy as np
import pytest
import torch

from oracle import oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M,N,K,G", [(65, 40, 256, 64), (96, 1000, 512, 128), (97, 64, 1536, 256),
                                     (128, 130, 768, 128), (129, 48, 512, 64), (192, 33, 1024, 256),
                                     (193, 24, 256, 128), (320, 16, 512, 64), (512, 40, 256, 128),
                                     (70, 4200, 256, 128), (130, 8200, 128, 128), (65, 8200, 256, 256),
                                     (131, 8208, 192, 64), (150, 8192, 96, 32)])
def test_w4a8_more_than_64_tokens(pkg, cuda, M, N, K, G):
    rng = np.random.default_rng(M + N + K + G)
    xq = rng.integers(-127, 128, size=(M, K + 16), dtype=np.int8)
    w = rng.integers(0, 256, size=(N, K // 2), dtype=np.uint8)
    ws = rng.uniform(1e-3, 1e-2, size=(N, K // G)).astype(np.float32)
    xs = rng.uniform(1e-3, 1e-1, size=M).astype(np.float32)
    bias = rng.standard_normal(N).astype(np.float16)
    qt = pkg.QTensor(torch.from_numpy(w).cuda(), torch.from_numpy(ws).cuda(),
                     scheme="per_group_i4", group_size=G, codebook="int4")
    y = pkg.gemm_quantized(torch.from_numpy(xq).cuda()[:, :K], torch.from_numpy(xs).cuda(), qt,
                           torch.from_numpy(bias).cuda())
    cols = np.unique(np.r_[0:min(N, 17), N - 1, rng.integers(0, N, 24)])
    yr = oracle.gemm_w4a8(np.ascontiguousarray(xq[:, :K]), xs, w[cols], ws[cols], G, bias[cols])
    yr = yr[0] if isinstance(yr, tuple) else yr
    assert np.array_equal(y.cpu().numpy()[:, cols].view(np.uint16), yr.view(np.uint16))
