"""The wide tiles of the experts' products: every height that the kernel has a loop for, chosen from the groups' sizes,
and more tiles than workgroups, against the products in 64 bits."""

import pytest
import torch
from test_grouped_wide_gpu import compare, listed, rand

from halite_amd.kernels import library, ops

pytestmark = pytest.mark.gpu

# 64 groups times four column tiles are one round of 256 compute units as long as no group is cut: tiles as high as the
# largest group, at both sides of 256, 288, 320 and 352 rows, beside lower ones
UNCUT = [352, 351, 321, 320, 319, 289, 288, 287, 257, 256, 225, 193, 161, 129, 65, 1] * 4
CASES = [
    (UNCUT, 1024, 128), (UNCUT, 1020, 256),
    ([321] * 64, 1024, 256), ([289] * 63 + [0], 1024, 128),
    ([353] * 64, 1024, 128),     # one row more than a tile has: two of 192
    ([2049] * 70, 256, 128),     # tiles of 320 rows at most, 490 of them for 480 workgroups
    ([700, 0, 1100, 3000], 2048, 256),
]


@pytest.mark.parametrize("gated", [False, True])
@pytest.mark.parametrize("counts, n, k", CASES)
def test_products_in_tiles_of_every_height(counts, n, k, gated):
    gpu = torch.device("cuda:0")
    rows, groups = sum(counts), len(counts)
    n = n // 2 // 4 * 4 if gated and n // 2 >= 256 else n
    assert library.core_library().hal_grouped_gemm_experts_kernel(rows, n, k, groups, int(gated)) == 2
    offsets, group_offsets, tile_offsets = listed(counts, gpu)
    tokens = rows // 2 + 1
    x = rand(tokens, k, seed=1).bfloat16().to(gpu)
    w = rand(groups, n, k, seed=2, scale=0.1).bfloat16().to(gpu)
    up = rand(groups, n, k, seed=4, scale=0.1).bfloat16().to(gpu) if gated else None
    pick = torch.randperm(rows, generator=torch.Generator().manual_seed(3)).int().to(gpu)
    dtype = torch.bfloat16 if gated else torch.float32
    y = torch.full((rows, n), 7.0, device=gpu, dtype=dtype)
    how = dict(w_up=up, limit=7.0, alpha=1.702) if gated else dict(row_dst=pick)
    ops.grouped_gemm(x, w, y, n_rows=rows, group_offsets=group_offsets, tile_offsets=tile_offsets, row_src=pick, src_div=2, **how)
    for g, (a, b) in enumerate(zip(offsets.tolist(), offsets.tolist()[1:])):
        xs, ws = x[pick[a:b].long() // 2].double(), w[g].double()
        want, size = xs @ ws.T, xs.abs() @ ws.abs().T
        if not gated:
            compare(y[pick[a:b].long()], want, (k, size), 0.0)
            continue
        us = up[g].double()
        gate, add = want.clamp(max=7.0), (xs @ us.T).clamp(-7.0, 7.0)
        result = gate * torch.sigmoid(1.702 * gate) * (add + 1.0)
        # (the gate's slope is at most 1.2, the sums' errors are those of ``compare``; bf16 rounds by 2^-8 at most)
        off = (k + 8) * 2.0**-23 * (1.2 * size * (add.abs() + 1.0) + (xs.abs() @ us.abs().T) * gate.abs())
        limit = off + (2.0**-8 + 1e-5) * result.abs() + 1e-6
        assert bool(((y[a:b].double() - result).abs() <= limit).all()), float(((y[a:b].double() - result).abs() / limit).max())
