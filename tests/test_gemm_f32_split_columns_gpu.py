"""Float32 products of prompts whose last tiles, or all, have fewer columns: the same bits as those of the wider tiles."""

import pytest
import torch

from halite_amd.kernels import ops


# all tiles the lower ones, K in two parts and in one, in turns; the wider for a round and the lower behind them, whose last one ends
# inside; three row tiles, of which a round takes no whole number of columns
@pytest.mark.gpu
@pytest.mark.parametrize("m, n, k", [(300, 6100, 2048), (300, 8200, 2048), (400, 8196, 4132), (300, 28700, 2052), (513, 16388, 2048), (770, 33000, 2048)])
def test_columns(m, n, k):
    gen = torch.Generator().manual_seed(n)
    a, w = torch.randn(m, k, generator=gen).cuda(), (torch.randn(n, k, generator=gen) * 0.02).cuda()
    got = ops.gemm_f32(a, w)
    want, size = a.double() @ w.double().T, a.double().abs() @ w.double().abs().T
    # (the bound of the tests of these tiles)
    assert bool(((got.double() - want).abs() <= (k // 32 + 16) * 2.0**-24 * size).all())
    assert torch.equal(ops.gemm_f32(a[:100].contiguous(), w), got[:100])  # tiles of 64 or 128 rows, 128 columns
