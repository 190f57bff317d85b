"""The experts' products of many groups, most of them without rows or with one: groups in runs of one to
eight a lane, against the products in 64 bits."""

import pytest
import torch

from halite_amd.kernels import library, ops

pytestmark = pytest.mark.gpu


def kernel_of(n_rows, n, k, n_groups, gated=False):
    return library.core_library().hal_grouped_gemm_experts_kernel(n_rows, n, k, n_groups, int(gated))


def some(n_groups, n_rows, seed):
    """So many rows to drawn groups, the first and the last and those around the lanes' runs among them."""
    gen = torch.Generator().manual_seed(seed)
    picks = torch.randint(0, n_groups, (n_rows,), generator=gen)
    edges = torch.tensor([g for g in (0, n_groups - 1, 63, 64, 65, 127, 128) if g < n_groups])
    picks[: len(edges)] = edges[:n_rows]
    return torch.bincount(picks, minlength=n_groups)


FEW, STREAM, WIDE, TILES = range(4)  # the kernels, as the library numbers them


# one lane a group and two, a last lane with part of a run and lanes without groups, the most groups there are;
# fewer rows than groups, and some rows each.  The last one: tiles for prompts
@pytest.mark.parametrize("n_groups, n_rows, plain, both", [
    (64, 100, STREAM, STREAM), (65, 40, FEW, STREAM), (86, 900, STREAM, STREAM), (129, 64, STREAM, STREAM), (300, 33, FEW, STREAM),
    (512, 1500, STREAM, STREAM), (512, 40, STREAM, STREAM), (150, 7500, WIDE, WIDE)])
@pytest.mark.parametrize("gated", [False, True])
def test_many_groups(n_groups, n_rows, plain, both, gated):
    n, k, top = 512, 256, 2
    assert kernel_of(n_rows, n, k, n_groups, gated) == (both if gated else plain)
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


def test_which_kernel():
    # 48 tokens, 4 of 16 experts; half of the chip's units have a tile, or fewer; a begun round with less than a row a group, and more
    assert kernel_of(192, 4096, 4096, 16) == STREAM
    assert kernel_of(4, 4096, 4096, 16) == FEW and kernel_of(4, 4608, 4096, 16) == STREAM
    assert kernel_of(40, 2048, 768, 256) == FEW and kernel_of(256, 4608, 4096, 16) == STREAM
    # that round over longer rows
    assert kernel_of(64, 768, 2048, 128, True) == STREAM and kernel_of(80, 512, 2048, 512, True) == STREAM and kernel_of(72, 512, 1536, 512, True) == STREAM
    # K of part of a line; many rows a group
    assert kernel_of(192, 4096, 4104, 16) == FEW and kernel_of(600, 4096, 4104, 16) == TILES
    # prompts: the wide tiles fill the chip or not, a round that has just begun, a long K
    assert kernel_of(9000, 4096, 4096, 16) == WIDE and kernel_of(18000, 4096, 1024, 64) == WIDE
    assert kernel_of(1600, 1024, 4096, 8, True) == STREAM and kernel_of(2048, 2816, 2048, 8, True) == TILES
    assert kernel_of(1600, 4096, 14336, 8) == TILES and kernel_of(3200, 2048, 256, 16) == STREAM
    # a short K has no streaming tiles
    assert kernel_of(1600, 1024, 128, 8) == WIDE and kernel_of(600, 192, 128, 8) == TILES


# rows of the groups at both sides of the wide tiles' heights (as in the test of those tiles), three times over, so that they fill the chip
EDGES = 3 * [0, 1, 33, 64, 65, 128, 129, 160, 0, 161, 192, 193, 224, 225, 255, 256, 257, 512, 513, 545, 2049, 0]


@pytest.mark.parametrize("n, k, kernel", [(260, 384, WIDE), (512, 256, WIDE), (132, 320, STREAM)])
def test_tiles_of_prompts(n, k, kernel):
    """Against 64 bits; and the bits of the tiles of 128, which a result that begins at an odd column gets."""
    ends = [0, *torch.tensor(EDGES).cumsum(0).tolist()]
    rows = ends[-1]
    assert kernel_of(rows, n, k, len(EDGES)) == kernel
    gen = torch.Generator().manual_seed(n)
    x = torch.randn(rows, k + 24, generator=gen).bfloat16().cuda()
    w = (0.1 * torch.randn(len(EDGES), n, k, generator=gen)).bfloat16().cuda()
    to = torch.randperm(rows, generator=gen).int().cuda()
    tiles = [0, *(-(-torch.tensor(EDGES) // ops.GROUP_TILE_ROWS)).cumsum(0).tolist()]
    y, general = (torch.full((rows, n + 12), 7.0, device="cuda") for _ in range(2))
    how = dict(n_rows=rows, x_col0=8, group_offsets=torch.tensor(ends).int().cuda(), tile_offsets=torch.tensor(tiles).int().cuda(), row_dst=to)
    ops.grouped_gemm(x, w, y, y_col0=4, **how)
    ops.grouped_gemm(x, w, general, y_col0=5, **how)
    assert bool((y[:, :4] == 7).all()) and bool((y[:, 4 + n :] == 7).all())
    assert torch.equal(y[:, 4 : 4 + n], general[:, 5 : 5 + n])
    for g, (a, b) in enumerate(zip(ends, ends[1:])):
        xs, ws = x[a:b, 8 : 8 + k].double(), w[g].double()
        limit = (k + 8) * 2.0**-23 * (xs.abs() @ ws.abs().T)  # (the matrix cores need not round to nearest)
        assert bool(((y[to[a:b].long(), 4 : 4 + n].double() - xs @ ws.T).abs() <= limit).all()), g


@pytest.mark.parametrize("rows", [4096, 4097])
def test_heads_of_one_step(rows):
    """Heads whose K is one step of the streaming tiles, at both sides of the rows from which tiles of 128 take them."""
    heads, n, k = 3, 68, 64
    gen = torch.Generator().manual_seed(rows)
    x = torch.randn(rows, heads * k, generator=gen).bfloat16().cuda()
    w = torch.randn(heads, n, k, generator=gen).bfloat16().cuda()
    y = torch.empty(rows, heads * n, device="cuda")
    ops.grouped_gemm(x, w, y, n_rows=rows, x_group_cols=k, y_group_cols=n)
    for h in range(heads):
        a, b = x[:, h * k : (h + 1) * k].double(), w[h].double()
        limit = (k + 8) * 2.0**-23 * (a.abs() @ b.abs().T)  # (the matrix cores need not round to nearest)
        assert bool(((y[:, h * n : (h + 1) * n].double() - a @ b.T).abs() <= limit).all())
