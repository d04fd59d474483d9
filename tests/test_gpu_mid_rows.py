"""The 64x128 prefill tile's automatic plans (65 to 512 rows split over K, and unsplit
where it fills two to three workgroups a CU) at the edges of their rules, with ragged
rows and columns: fp16 outputs and accumulators bit for bit against the oracle on
sampled rows, through the workspace entry and without a workspace."""
import numpy as np
import pytest
import torch

from oracle import oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M,N,K", [(65, 512, 3072), (65, 1000, 3072), (128, 2048, 3200),
                                   (128, 24576, 3072), (129, 1024, 3072), (256, 2048, 4096),
                                   (333, 1536, 4608), (512, 1024, 3072), (300, 4000, 8192),
                                   (577, 7000, 1024), (700, 8900, 1152)])
def test_mid_rows(pkg, cuda, M, N, K):
    g = torch.Generator(device="cuda").manual_seed(M + N + K)
    q = torch.randint(-127, 128, (N, K), generator=g, dtype=torch.int8, device="cuda")
    xq = torch.randint(-127, 128, (M, K), generator=g, dtype=torch.int8, device="cuda")
    s = torch.rand(N, generator=g, device="cuda") * 0.01
    xs = torch.rand(M, generator=g, device="cuda") * 0.1
    bias = torch.randn(N, generator=g, device="cuda").half()
    qt = pkg.QTensor(q, s, scheme="per_row_i8")
    rows = np.unique(np.r_[0, 63, 64, M - 1, np.random.default_rng(M).integers(0, M, 12)])
    accr = oracle.gemm_i8(xq.cpu().numpy()[rows], q.cpu().numpy())
    yr = oracle.dequant_f16(accr, xs.cpu().numpy()[rows], s.cpu().numpy(),
                            bias.cpu().numpy()).view(np.uint16)
    for _ in range(2):  # the second call finds the first one's workspace
        y, acc = pkg.gemm_w8a8(xq, xs, qt, bias, want_acc=True)
        y2 = pkg.gemm_w8a8(xq, xs, qt, bias)
        assert np.array_equal(acc.cpu().numpy()[rows], accr)
        assert np.array_equal(y.cpu().numpy()[rows].view(np.uint16), yr)
        assert torch.equal(y2, y)
