"""W8A8 GEMMs whose K is no multiple of 64 or 128 (a tensor-parallel shard's
width) and rows that are only 4-byte aligned: the skinny kernel's last K % 64
bytes and the 32x32x32 tile kernel's ragged K steps, dense and over expert
segments.  Integer accumulation is exact, so every output is bit for bit the
oracle's."""
import numpy as np
import pytest
import torch

from oracle import oracle

pytestmark = pytest.mark.gpu


# K: below one 64-byte unit, one byte quad past or short of a unit, of a 128-byte
# step and of an even number of steps, 16-byte aligned rows and 4-byte aligned ones
@pytest.mark.parametrize("K", [4, 60, 68, 124, 132, 192, 252, 260, 368, 1376, 2084])
@pytest.mark.parametrize("M,N", [(1, 33), (16, 100), (17, 16), (33, 130), (64, 31), (65, 127),
                                 (129, 200), (300, 257)])
def test_ragged_k(pkg, cuda, M, N, K):
    """M crosses every row block of the skinny kernel and enters the tile kernel's
    128-, 256- and 64-row tiles; `lda` puts the activation rows 4 bytes apart from
    16-byte alignment in half of the cases."""
    rng = np.random.default_rng(M * 7919 + N * 31 + K)
    pad = 4 if (M + K) % 8 else 0
    xq = rng.integers(-127, 128, size=(M, K + pad), dtype=np.int8)
    q = rng.integers(-127, 128, size=(N, K), dtype=np.int8)
    xs = rng.uniform(0.001, 0.1, size=M).astype(np.float32)
    s = rng.uniform(0.001, 0.02, size=N).astype(np.float32)
    bias = rng.standard_normal(N).astype(np.float16)
    qt = pkg.QTensor(torch.from_numpy(q).cuda(), torch.from_numpy(s).cuda(), scheme="per_row_i8")
    xd = torch.from_numpy(xq).cuda()[:, :K]
    args = (xd, torch.from_numpy(xs).cuda(), qt, torch.from_numpy(bias).cuda())
    y, acc = pkg.gemm_w8a8(*args, want_acc=True)
    y2 = pkg.gemm_w8a8(*args)
    torch.cuda.synchronize()
    accr = oracle.gemm_i8(np.ascontiguousarray(xq[:, :K]), q)
    assert np.array_equal(acc.cpu().numpy(), accr)
    yr = oracle.dequant_f16(accr, xs, s, bias).view(np.uint16)
    assert np.array_equal(y.cpu().numpy().view(np.uint16), yr)
    assert np.array_equal(y2.cpu().numpy().view(np.uint16), yr)


def test_ragged_k_tall(pkg, cuda):
    """Enough row tiles that the 256x128 ragged tile is chosen."""
    M, N, K = 2600, 2090, 340
    rng = np.random.default_rng(5)
    xq = rng.integers(-127, 128, size=(M, K), dtype=np.int8)
    q = rng.integers(-127, 128, size=(N, K), dtype=np.int8)
    xs, s = np.full(M, 0.01, np.float32), rng.uniform(0.001, 0.02, size=N).astype(np.float32)
    qt = pkg.QTensor(torch.from_numpy(q).cuda(), torch.from_numpy(s).cuda(), scheme="per_row_i8")
    y = pkg.gemm_w8a8(torch.from_numpy(xq).cuda(), torch.from_numpy(xs).cuda(), qt)
    yr = oracle.dequant_f16(oracle.gemm_i8(xq, q), xs, s)
    assert np.array_equal(y.cpu().numpy().view(np.uint16), yr.view(np.uint16))


@pytest.mark.parametrize("K", [68, 172, 192, 368])
@pytest.mark.parametrize("T", [3, 40, 400])
def test_ragged_k_grouped(pkg, cuda, T, K):
    """Expert segments: the skinny kernel (T = 3), 64- and 128-row tiles."""
    E, k, N = 8, 2, 130
    rng = np.random.default_rng(T + K)
    topi = np.stack([rng.permutation(E - 1)[:k] for _ in range(T)]).astype(np.int32)  # one empty
    aq = rng.integers(-127, 128, size=(T, K), dtype=np.int8)
    as_ = rng.uniform(0.001, 0.1, size=T).astype(np.float32)
    w = rng.integers(-127, 128, size=(E, N, K), dtype=np.int8)
    ws = rng.uniform(0.001, 0.02, size=(E, N)).astype(np.float32)
    seg, rt, _ = pkg.moe_sort(torch.from_numpy(topi).cuda(), E)
    y, acc = pkg.gemm_w8a8_grouped(torch.from_numpy(aq).cuda(), torch.from_numpy(as_).cuda(),
                                   torch.from_numpy(w).cuda(), torch.from_numpy(ws).cuda(), seg,
                                   T * k, row_index=rt, want_acc=True)
    torch.cuda.synchronize()
    seg_r, rt_r, _, _ = oracle.moe_sort(topi, E)
    yr, accr = oracle.grouped_w8a8_f16(aq, as_, w, ws, seg_r, row_index=rt_r, want_acc=True)
    assert np.array_equal(acc.cpu().numpy(), accr)
    assert np.array_equal(y.cpu().numpy().view(np.uint16), yr.view(np.uint16))
