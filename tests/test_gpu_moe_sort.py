"""The routing sort at the edges of its wave and register shares: 2048 ids (4 or more
waves), 256 experts (16 or 8 waves), 16384 or 8192 ids (kept in registers or read again),
ragged ends, an id array that is only 4-byte aligned, and ids outside [0, E).  Whole
numbers: exact."""
import numpy as np
import pytest
import torch

from oracle import oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T,k,E", [(1, 1, 1), (2047, 1, 7), (2048, 1, 5), (2049, 1, 5), (683, 3, 16),
                                   (5461, 6, 64), (32768, 1, 3), (32769, 1, 3), (20011, 2, 130),
                                   (16384, 1, 256), (16385, 1, 256), (2048, 1, 257),
                                   (2049, 1, 257), (4096, 2, 300), (8193, 1, 300), (3000, 8, 512)])
def test_sort_edges(pkg, cuda, T, k, E):
    rng = np.random.default_rng(T + E)
    ids = rng.integers(0, E, size=(T + 1, k)).astype(np.int32)
    d = torch.from_numpy(ids).cuda()[1:]  # 4 * k bytes past the allocation's alignment
    seg, rt, pos = pkg.moe_sort(d, E)
    torch.cuda.synchronize()
    seg_r, rt_r, _, pos_r = oracle.moe_sort(ids[1:].astype(np.int64), E)
    assert np.array_equal(seg.cpu().numpy(), seg_r)
    assert np.array_equal(rt.cpu().numpy(), rt_r)
    assert np.array_equal(pos.cpu().numpy(), pos_r)


@pytest.mark.parametrize("T", [100, 3000])
def test_sort_ids_out_of_range(pkg, cuda, T):
    """An id outside [0, E) has no row: pos -1, and the others sort as without it."""
    E, k = 12, 2
    rng = np.random.default_rng(T)
    ids = rng.integers(-2, E + 2, size=(T, k)).astype(np.int32)
    seg, rt, pos = pkg.moe_sort(torch.from_numpy(ids).cuda(), E)
    torch.cuda.synchronize()
    flat = ids.reshape(-1)
    ok = np.flatnonzero((flat >= 0) & (flat < E))
    order = ok[np.argsort(flat[ok], kind="stable")]
    want = np.full(T * k, -1, np.int32)
    want[order] = np.arange(order.size)
    assert np.array_equal(pos.cpu().numpy().reshape(-1), want)
    assert np.array_equal(rt.cpu().numpy()[:order.size], order // k)
    assert np.array_equal(seg.cpu().numpy(),
                          np.searchsorted(flat[order], np.arange(E + 1), side="left"))


def test_sort_most_ids(pkg, cuda):
    """The largest T * k that the entry point takes: no count on the way passes 2^31.
    Three ids of expert 1 among ids of expert 0, looked at where the rows change."""
    T = 2**31 - 1
    at = [5, 2**30, T - 2]
    ids = torch.zeros(T, 1, dtype=torch.int32, device="cuda")
    for i in at:
        ids[i] = 1
    seg, rt, pos = pkg.moe_sort(ids, 2)
    torch.cuda.synchronize()
    del ids
    assert seg.tolist() == [0, T - 3, T]
    assert rt[:7].tolist() == [0, 1, 2, 3, 4, 6, 7]
    assert rt[T - 5:].tolist() == [T - 3, T - 1] + at
    assert pos[:7, 0].tolist() == [0, 1, 2, 3, 4, T - 3, 5]
    assert pos[2**30 - 1:2**30 + 2, 0].tolist() == [2**30 - 2, T - 2, 2**30 - 1]
    assert pos[T - 3:, 0].tolist() == [T - 5, T - 1, T - 4]
    del rt, pos
    torch.cuda.empty_cache()
