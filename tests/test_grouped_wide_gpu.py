"""The experts' products: of prompts (tiles of up to 256 rows whose height follows the groups' sizes, and
streaming tiles where those would not fill the chip) and of few rows a group (streaming tiles, and the
kernel for few rows), against the products in 64 bits."""

import pytest
import torch

from halite_amd.kernels import ops

pytestmark = pytest.mark.gpu


@pytest.fixture
def gpu():
    return torch.device("cuda:0")


# rows of the groups: none, one, at both sides of every height that the kernel has a loop for (64, 128, 160,
# 192, 224, 256 rows), of a second, third and ninth tile (a panel of eight and one more), and a group whose
# equal heights in steps of 32 leave its last tile short
EDGES = [0, 1, 33, 64, 65, 128, 129, 160, 0, 161, 192, 193, 224, 225, 255, 256, 257, 512, 513, 545, 2049, 0]
# fewer than 48 a group on average: the streaming tiles (the long list of single rows: the kernel for few rows); none, one, at both sides of 32 and 64 rows, several tiles
FEW = [0, 1, 31, 32, 33, 0, 63, 64, 65, 0, 0, 97, 129, 2, 16, 17, 0, 0, 200, 0]


def listed(counts, device):
    offsets = torch.tensor([0] + counts).cumsum(0)
    tiles = torch.tensor([0] + [-(-c // ops.GROUP_TILE_ROWS) for c in counts]).cumsum(0)
    return offsets, offsets.int().to(device), tiles.int().to(device)


def rand(*shape, seed, scale=1.0):
    return scale * torch.randn(*shape, generator=torch.Generator().manual_seed(seed))


def compare(got, want, size, result_rounding):
    """``size``: the products' terms without their signs, summed.  A float32 sum of K terms is off by at
    most K rounding errors of that sum (2^-23: the matrix cores need not round to nearest)."""
    k, magnitude = size
    limit = (k + 8) * 2.0**-23 * magnitude + result_rounding * want.abs() + 1e-30
    assert bool(((got.double() - want).abs() <= limit).all()), float(((got.double() - want).abs() / limit).max())


@pytest.mark.parametrize("counts, n, k", [(EDGES, 256, 128), (EDGES, 260, 384), (EDGES, 768, 256), ([300] * 70, 256, 128),
                                          (FEW, 128, 256), (FEW, 132, 320), (FEW, 300, 384), ([1] * 3 + [0] * 80 + [5] * 3, 256, 448)])
def test_down_products_scatter_float32_rows(gpu, counts, n, k):
    """Rows and results with strides of their own, results at scattered rows, more groups than lanes of a wave."""
    rows = sum(counts)
    offsets, group_offsets, tile_offsets = listed(counts, gpu)
    x = rand(rows, k + 24, seed=1).bfloat16().to(gpu)
    w = rand(len(counts), n, k, seed=2, scale=0.1).bfloat16().to(gpu)
    to = torch.randperm(rows, generator=torch.Generator().manual_seed(3)).int().to(gpu)
    y = torch.full((rows, n + 12), 7.0, device=gpu)
    ops.grouped_gemm(x, w, y, n_rows=rows, x_col0=8, y_col0=4, group_offsets=group_offsets, tile_offsets=tile_offsets, row_dst=to)
    assert bool((y[:, :4] == 7).all()) and bool((y[:, 4 + n :] == 7).all())
    for g, (a, b) in enumerate(zip(offsets.tolist(), offsets.tolist()[1:])):
        xs, ws = x[a:b, 8 : 8 + k].double(), w[g].double()
        compare(y[to[a:b].long(), 4 : 4 + n], xs @ ws.T, (k, xs.abs() @ ws.abs().T), 0.0)


@pytest.mark.parametrize("act", ["gated", "relu_squared"])
@pytest.mark.parametrize("counts, n, k", [(EDGES, 256, 128), (EDGES, 388, 256), (FEW, 128, 256), (FEW, 200, 320), (FEW, 388, 384)])
def test_up_products_gather_rows(gpu, act, counts, n, k):
    """Rows gathered through the sorted list, the activations in the epilogue, bf16 results."""
    top = 2
    rows = sum(counts)
    offsets, group_offsets, tile_offsets = listed(counts, gpu)
    tokens = -(-rows // top)
    x = rand(tokens, k, seed=4).bfloat16().to(gpu)
    w, up = (rand(len(counts), n, k, seed=5 + i, scale=0.15).bfloat16().to(gpu) for i in range(2))
    order = torch.randperm(rows, generator=torch.Generator().manual_seed(6)).int().to(gpu)
    y = torch.empty((rows, n), dtype=torch.bfloat16, device=gpu)
    how = dict(w_up=up, limit=1.5, alpha=1.702) if act == "gated" else dict(relu_squared=True)
    ops.grouped_gemm(x, w, y, n_rows=rows, group_offsets=group_offsets, tile_offsets=tile_offsets, row_src=order, src_div=top, **how)
    for g, (a, b) in enumerate(zip(offsets.tolist(), offsets.tolist()[1:])):
        xs = x[order[a:b].long() // top].double()
        z = xs @ w[g].double().T
        size = xs.abs() @ w[g].abs().double().T
        if act == "gated":
            u = xs @ up[g].double().T
            gate, shifted = z.clamp(max=1.5), u.clamp(-1.5, 1.5) + 1
            want = gate * torch.sigmoid(1.702 * gate) * shifted
            # both factors move at most as their products do (the gate's slope is below 1.2); the exponential is good to 2^-20
            size = 1.2 * size * shifted.abs() + (xs.abs() @ up[g].abs().double().T) * gate.abs()
        else:
            want = torch.relu(z) ** 2
            size = 2 * size * torch.relu(z) + size * size * k * 2.0**-23
        compare(y[a:b], want, (k, size), 2.0**-8 + 2.0**-18)


def test_a_row_does_not_depend_on_its_neighbours(gpu):
    """The same rows in groups of other sizes, and with a K of another number of steps (the added columns are
    zeros), give the same bits."""
    n, k, rows = 256, 256, 700
    x, w = rand(rows, k, seed=7).bfloat16().to(gpu), rand(1, n, k, seed=8, scale=0.1).bfloat16().to(gpu)
    whole = torch.empty((rows, n), device=gpu)
    _, go, to = listed([rows], gpu)
    ops.grouped_gemm(x, w, whole, n_rows=rows, group_offsets=go, tile_offsets=to)
    counts = [200, 3, 130, 367]
    parts = torch.empty((rows, n), device=gpu)
    _, go, to = listed(counts, gpu)
    ops.grouped_gemm(x, w.expand(4, n, k).contiguous(), parts, n_rows=rows, group_offsets=go, tile_offsets=to)
    assert torch.equal(whole, parts)
    wide = torch.zeros((rows, k + 64), dtype=torch.bfloat16, device=gpu)
    wide[:, :k] = x
    ww = torch.zeros((4, n, k + 64), dtype=torch.bfloat16, device=gpu)
    ww[:, :, :k] = w
    other = torch.empty((rows, n), device=gpu)
    ops.grouped_gemm(wide, ww, other, n_rows=rows, group_offsets=go, tile_offsets=to)
    assert torch.equal(whole, other)
