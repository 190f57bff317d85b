"""Products in groups over rows that overlap in memory: one row that stands for all, and rows a few
elements apart, by every kernel that loads its rows straight into LDS."""

import pytest
import torch

from halite_amd.kernels import ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("apart, col0", [(0, 0), (0, 8), (8, 8)])
@pytest.mark.parametrize("groups, rows", [("heads", 40), ("experts", 60), ("experts", 400)])  # the last two: streaming and wide tiles
def test_overlapping_rows(groups, rows, apart, col0):
    g, n, k = 3, 768, 256
    gen = torch.Generator().manual_seed(rows)
    width = col0 + (g * k if groups == "heads" else k)
    memory = torch.randn(rows * 8 + width, generator=gen).bfloat16().cuda()
    w = torch.randn(g, n, k, generator=gen).bfloat16().cuda()
    x = memory.as_strided((rows, width), (apart, 1))
    if groups == "heads":
        y = torch.zeros(rows, g * n, device="cuda")
        ops.grouped_gemm(x, w, y, n_rows=rows, x_group_cols=k, x_col0=col0, y_group_cols=n)
        parts = [(x[:, col0 + h * k : col0 + (h + 1) * k], w[h], y[:, h * n : (h + 1) * n]) for h in range(g)]
    else:
        counts = torch.tensor([rows // 2, 1, rows - rows // 2 - 1])
        ends = [0, *counts.cumsum(0).tolist()]
        offsets = torch.tensor(ends, dtype=torch.int32, device="cuda")
        tiles = torch.tensor([0, *(-(-counts // ops.GROUP_TILE_ROWS)).cumsum(0).tolist()], dtype=torch.int32, device="cuda")
        y = torch.zeros(rows, n, device="cuda")
        ops.grouped_gemm(x, w, y, n_rows=rows, x_col0=col0, group_offsets=offsets, tile_offsets=tiles)
        parts = [(x[a:b, col0:], w[e], y[a:b]) for e, (a, b) in enumerate(zip(ends, ends[1:]))]
    for xs, ws, got in parts:
        a, b = xs.double(), ws.double()
        # a sum of k exact products in 32 bits (the matrix cores need not round to nearest)
        assert bool(((got.double() - a @ b.T).abs() <= (k + 8) * 2.0**-23 * (a.abs() @ b.abs().T)).all())
