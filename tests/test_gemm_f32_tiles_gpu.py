"""The float32 product in tiles of 128, 64 and 32 columns: sizes at which each is launched, with rows and
columns that end inside a tile, against the product in 64 bits."""

import pytest
import torch

from halite_amd.kernels import library, ops

pytestmark = pytest.mark.gpu


# tiles of 32 in one, three and five rounds, of 64 in one, two and three, and of 128 in full rounds: a last tile of one row more
# than half of its waves take, of so few that half of them have none, and of nearly all
@pytest.mark.parametrize("m, n, k, columns", [(130, 4000, 36, 32), (300, 4100, 1028, 64), (500, 4090, 544, 64), (260, 28004, 64, 64),
                                              (700, 4033, 96, 32), (1030, 4161, 512, 32), (1500, 4090, 1028, 64),
                                              (449, 16384, 132, 128), (400, 16378, 1060, 128), (1000, 8190, 100, 128), (2000, 4090, 516, 128)])
def test_tiles(m, n, k, columns):
    assert library.core_library().hal_gemm_f32_columns(m, n) == columns
    gen = torch.Generator().manual_seed(m)
    a, w = torch.randn(m, k, generator=gen).cuda(), torch.randn(n, k, generator=gen).cuda()
    got = ops.gemm_f32(a, w).double()
    want, size = a.double() @ w.double().T, a.double().abs() @ w.double().abs().T
    # stretches of 512 summed from nothing, then added up: at most as many roundings one on the other
    assert bool(((got - want).abs() <= (min(k, 512) + k // 512 + 2) * 2.0**-24 * size).all())
    # a row's result is its own, whatever tile it is in
    part = ops.gemm_f32(a[: m - 1].contiguous(), w[: n // 2].contiguous()).double()
    assert torch.equal(part, got[: m - 1, : n // 2])
