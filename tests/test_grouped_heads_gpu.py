"""The product of heads in streaming tiles: rows and columns around the tiles' edges, one step of K to
several turns through the buffers, with and without gates, against the products in 64 bits."""

import pytest
import torch

from halite_amd.kernels import ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows", [17, 32, 33, 64, 65, 200])
@pytest.mark.parametrize("k, n", [(64, 4), (128, 192), (192, 128), (256, 132), (320, 260)])
@pytest.mark.parametrize("gate_of, dtype", [(None, torch.bfloat16), (None, torch.float32), ("column", torch.bfloat16), ("head", torch.float32)])
def test_heads(rows, k, n, gate_of, dtype):
    heads, x0, y0 = 3, 8, 4
    xs, ys = x0 + k + 16, y0 + n + 8
    gen = torch.Generator().manual_seed(rows * k + n)
    x = torch.randn(rows, heads * xs, generator=gen).bfloat16().cuda()
    w = torch.randn(heads, n, k, generator=gen).bfloat16().cuda()
    gate = None if gate_of is None else torch.randn(rows, 3 + (heads * ys if gate_of == "column" else heads), generator=gen).cuda()[:, 3:]
    y = torch.full((rows, heads * ys), 7.0, dtype=dtype, device="cuda")
    ops.grouped_gemm(x, w, y, n_rows=rows, x_group_cols=xs, x_col0=x0, y_group_cols=ys, y_col0=y0, gate=gate, gate_per_group=gate_of == "head")
    want, bound = torch.full((rows, heads * ys), 7.0, dtype=torch.float64, device="cuda"), torch.zeros(rows, heads * ys, dtype=torch.float64, device="cuda")
    for h in range(heads):
        a, b = x[:, h * xs + x0 : h * xs + x0 + k].double(), w[h].double()
        at = slice(h * ys + y0, h * ys + y0 + n)
        by = 1.0
        if gate is not None:
            by = torch.sigmoid((gate[:, h * ys : h * ys + n] if gate_of == "column" else gate[:, h : h + 1]).double())
        want[:, at] = a @ b.T * by
        # a sum of k exact products in 32 bits, and a sigmoid to some units in the last place
        bound[:, at] = (k + 8) * 2.0**-24 * (a.abs() @ b.abs().T) * by
    if dtype == torch.bfloat16:
        bound += 2.0**-8 * (want.abs() + bound) * (bound > 0)
    assert bool(((y.double() - want).abs() <= bound).all())
