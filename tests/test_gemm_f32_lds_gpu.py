"""Float32 products of more rows than 96 (32 of wide matrices) whose operands go straight into LDS: every width of the tiles, ends of K inside
a stage, and fewer stages than buffers."""

import pytest
import torch

from halite_amd.kernels import library, ops

pytestmark = pytest.mark.gpu


# one tile and one more row or column than tiles have, K of one number group, of one stage and a little more, of two
# stretches and a little more; tiles of 96 in all but one of a round's places and in all of them
@pytest.mark.parametrize("m, n, k, columns", [(129, 4090, 4, 32), (256, 4096, 32, 32), (129, 4097, 36, 64), (384, 5441, 100, 96),
                                              (500, 6048, 68, 96), (512, 6144, 1060, 96), (640, 4033, 132, 96),
                                              (1500, 4090, 64, 64), (512, 16384, 60, 128), (1024, 8100, 576, 128),
                                              (33, 16384, 96, 64), (64, 28676, 1028, 64), (97, 16257, 36, 64)])
def test_every_width(m, n, k, columns):
    assert library.core_library().hal_gemm_f32_columns(m, n) == columns
    gen = torch.Generator().manual_seed(m + k)
    a, w = torch.randn(m, k, generator=gen).cuda(), torch.randn(n, k, generator=gen).cuda()
    got = ops.gemm_f32(a, w).double()
    a, w = a.double(), w.double()
    # stretches of 512 summed from nothing, then added up: at most as many roundings one on the other
    assert bool(((got - a @ w.T).abs() <= (min(k, 512) + k // 512 + 2) * 2.0**-24 * (a.abs() @ w.abs().T)).all())
