"""The experts' products of many groups, most of them without rows or with one: groups in runs of one to
eight a lane, against the products in 64 bits."""

import pytest
import torch

from halite_amd.kernels import ops

pytestmark = pytest.mark.gpu


def some(n_groups, n_rows, seed):
    """So many rows to drawn groups, the first and the last and those around the lanes' runs among them."""
    gen = torch.Generator().manual_seed(seed)
    picks = torch.randint(0, n_groups, (n_rows,), generator=gen)
    edges = torch.tensor([g for g in (0, n_groups - 1, 63, 64, 65, 127, 128) if g < n_groups])
    picks[: len(edges)] = edges[:n_rows]
    return torch.bincount(picks, minlength=n_groups)


# one lane a group and two, a last lane with part of a run and lanes without groups, the most groups there are;
# fewer rows than groups, and some rows each.  The last one: tiles for prompts
@pytest.mark.parametrize("n_groups, n_rows", [(64, 100), (65, 40), (86, 900), (129, 64), (300, 33), (512, 1500), (512, 40), (130, 6600)])
@pytest.mark.parametrize("gated", [False, True])
def test_many_groups(n_groups, n_rows, gated):
    n, k, top = 512, 256, 2
    counts = some(n_groups, n_rows, n_groups)
    ends = [0, *counts.cumsum(0).tolist()]
    dev = lambda t: t.int().cuda()  # noqa: E731
    offsets, tiles = dev(torch.tensor(ends)), dev(torch.tensor([0, *(-(-counts // ops.GROUP_TILE_ROWS)).cumsum(0).tolist()]))
    gen = torch.Generator().manual_seed(n_rows)
    x = torch.randn(-(-n_rows // top), k, generator=gen).bfloat16().cuda()
    w, up = ((0.1 * torch.randn(n_groups, n, k, generator=gen)).bfloat16().cuda() for _ in range(2))
    order = dev(torch.randperm(n_rows, generator=gen))
    y = torch.full((n_rows, n), 7.0, device="cuda")
    how = dict(w_up=up, limit=float("inf"), alpha=1.0, up_shift=0.0) if gated else {}
    ops.grouped_gemm(x, w, y, n_rows=n_rows, group_offsets=offsets, tile_offsets=tiles, row_src=order, src_div=top, **how)
    bit = 2.0**-23  # (the matrix cores need not round to nearest)
    for g, (a, b) in enumerate(zip(ends, ends[1:])):
        if a == b:
            continue
        xs = x[order[a:b].long() // top].double()
        z, size = xs @ w[g].double().T, xs.abs() @ w[g].double().abs().T
        want, limit = z, (k + 8) * bit * size
        if gated:
            u, size_u = xs @ up[g].double().T, xs.abs() @ up[g].double().abs().T
            want = z * torch.sigmoid(z) * u
            # the gate's slope is below 1.2; the exponential is good to 2^-20
            limit = (k + 8) * bit * (1.2 * size * u.abs() + size_u * z.abs()) + 2.0**-18 * want.abs() + (k * bit) ** 2 * size * size_u
        assert bool(((y[a:b].double() - want).abs() <= limit).all()), g
