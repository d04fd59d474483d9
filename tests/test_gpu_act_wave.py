"""act_and_mul_quant with one wave per row: 256 rows and more of up to 512 elements, 1536
of up to 768 and 3072 of up to 1024, at the edges of these and of the lanes' 8-byte
chunks, with a ragged last workgroup and rows of zeros, NaN and infinities; int8 rows and
scales bit for bit against the oracle."""
import numpy as np
import pytest
import torch

from oracle import oracle as o

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("act", ["silu", "gelu_tanh"])
@pytest.mark.parametrize("M,I", [(256, 8), (257, 248), (258, 256), (259, 264), (256, 512),
                                 (300, 768), (257, 1024), (256, 1032), (255, 768),
                                 (1535, 512), (1536, 520), (1537, 768), (1536, 776), (3071, 1024),
                                 (3072, 776), (3073, 1024), (3072, 1032)])
def test_act_quant_wave_rows(pkg, act, M, I):
    rng = np.random.default_rng(M + I)
    x = (rng.standard_normal((M, 2 * I)) * 4).astype(np.float16)
    x[3] = 0
    x[5, 0], x[6, I], x[7, 0] = np.nan, np.inf, -np.inf
    x[8] = 6e-8
    x[9, :I] = 60000
    xq, xs = pkg.act_and_mul_quant(torch.from_numpy(x).cuda(), act)
    q, s = o.act_and_mul_quant_f16(x, act)
    assert np.array_equal(xq.cpu().numpy(), q)
    got, nan = xs.cpu().numpy(), np.isnan(s)
    assert np.array_equal(np.isnan(got), nan)
    assert np.array_equal(got[~nan].view(np.uint32), s[~nan].view(np.uint32))
