"""The float32 product in tiles of 128, 64 and 32 columns: sizes at which each is chosen, with rows and
columns that end inside a tile, against the product in 64 bits."""

import pytest
import torch

from halite_amd.kernels import ops

pytestmark = pytest.mark.gpu


# 130 x 4,000: tiles of 32 (one round); 300 x 4,100 and 500 x 4,090: of 64 (one round); 260 x 28,004: of
# 128; 700 x 4,033: of 32 (three rounds); 1,030 x 4,161: of 64 (three rounds)
@pytest.mark.parametrize("m, n, k", [(130, 4000, 36), (300, 4100, 1028), (500, 4090, 544), (260, 28004, 64), (700, 4033, 96), (1030, 4161, 512)])
def test_tiles(m, n, k):
    gen = torch.Generator().manual_seed(m)
    a, w = torch.randn(m, k, generator=gen).cuda(), torch.randn(n, k, generator=gen).cuda()
    got = ops.gemm_f32(a, w).double()
    want, size = a.double() @ w.double().T, a.double().abs() @ w.double().abs().T
    # stretches of 512 summed from nothing, then added up: at most as many roundings one on the other
    assert bool(((got - want).abs() <= (min(k, 512) + k // 512 + 2) * 2.0**-24 * size).all())
    # a row's result is its own, whatever tile it is in
    part = ops.gemm_f32(a[: m - 1].contiguous(), w[: n // 2].contiguous()).double()
    assert torch.equal(part, got[: m - 1, : n // 2])
