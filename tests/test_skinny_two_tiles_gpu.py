"""Products of 9 to 16 rows whose workgroups take two tiles of the weight: against float64, and against the same rows in calls of
eight, which take one tile each."""

import pytest
import torch

pytestmark = pytest.mark.gpu


def rows_of(n, k, seed, gpu, scale=1.0):
    return (torch.randn((n, k), generator=torch.Generator().manual_seed(seed)) * scale).bfloat16().to(gpu)


def within_a_sum(got, want, size, k, what):
    """A sum of k products of bf16 numbers in float32 (a rounding of at most 2^-23 of what has been summed in size for each instruction's 32
    and each wave's part), then one rounding to bf16."""
    bound = size * (k / 32 + 32) * 2.0 ** -23 + want.abs() * 2.0 ** -8
    assert bool(((got.double() - want).abs() <= bound).all()), what


@pytest.mark.parametrize("m", [8, 9, 12, 13, 16])
@pytest.mark.parametrize("n, k", [
    (4096, 520), (4105, 264), (7168, 256), (7176, 256),  # 256, 257 (the last one of 9 rows), 448 and 449 tiles
    (8192, 128), (16384, 64),  # from 13 rows on by rounds
])
def test_plain_and_scaled(gpu, m, n, k):
    from halite_amd.kernels import ops

    x, w = rows_of(m, k, m, gpu), rows_of(n, k, n, gpu)
    tiled = ops.tile_weight(w)
    want, size = x.double() @ w.double().T, x.double().abs() @ w.double().abs().T
    got = ops.gemm_bf16_skinny(x, tiled, tiled_shape=(n, k), out_dtype=torch.float32)
    within_a_sum(got, want, size, k, "float32")
    within_a_sum(ops.gemm_bf16_skinny(x, tiled, tiled_shape=(n, k)), want, size, k, "bf16")
    halves = torch.cat([ops.gemm_bf16_skinny(part.contiguous(), tiled, tiled_shape=(n, k), out_dtype=torch.float32) for part in x.split(8)])
    within_a_sum(got, halves.double(), 2 * size, k, "calls of eight rows")
    # sums of squares of which row r's are k 4^(r % 3): the product is halved r % 3 times, exactly but for eps
    parts = torch.zeros((5, 16), device=gpu)
    parts[3, :m] = k * 4.0 ** (torch.arange(m, device=gpu) % 3)
    rows = ops.NormedRows(x, parts, 1e-12, torch.ones(k, device=gpu))
    scale = 2.0 ** -(torch.arange(m, device=gpu) % 3).double()[:, None]
    within_a_sum(ops.gemm_bf16_skinny_norm(rows, tiled, (n, k)), want * scale, size * scale, k, "scaled")


@pytest.mark.parametrize("m", [9, 13, 16])
@pytest.mark.parametrize("n, k", [(4112, 264), (5504, 512), (8192, 64), (14336, 64), (11000, 64)])
def test_gated(gpu, m, n, k):
    from halite_amd.kernels import ops

    x, w, up = rows_of(m, k, m, gpu), rows_of(n, k, 1, gpu, 0.05), rows_of(n, k, 2, gpu)
    t, t_up = ops.tile_weight(w), ops.tile_weight(up)
    g, u = x.double() @ w.double().T, x.double() @ up.double().T
    size_g, size_u = x.double().abs() @ w.double().abs().T, x.double().abs() @ up.double().abs().T
    want = u * g * torch.sigmoid(g)
    # silu's slope is at most 1.1; its own float32 steps are a few of 2^-23 of |g|
    steps = (k / 32 + 32) * 2.0 ** -23
    bound = (size_u * (g * torch.sigmoid(g)).abs() + 1.1 * size_g * u.abs()) * steps + want.abs() * 2.0 ** -7.9 + 1e-6
    assert bool(((ops.gemm_bf16_skinny(x, t, w_up=t_up, tiled_shape=(n, k)).double() - want).abs() <= bound).all())
    parts = torch.full((7, 16), k / 7.0, device=gpu)
    rows = ops.NormedRows(x, parts, 1e-12, torch.ones(k, device=gpu))
    got = ops.gemm_bf16_skinny_norm(rows, t, (n, k), w_up_tiled=t_up)
    assert bool(((got.double() - want).abs() <= bound + want.abs() * 2.0 ** -20).all())


@pytest.mark.parametrize("m", [9, 12, 16])
@pytest.mark.parametrize("H, K, D, width", [(24, 8, 128, 96), (33, 4, 112, 136), (257, 1, 16, 64), (48, 8, 128, 64)])
@pytest.mark.parametrize("normed", [False, True])
def test_rotated_and_appended(gpu, m, H, K, D, width, normed):
    """320, 287, 259 (the last workgroup's second tile is past the end) and 512 tiles: as two calls of fewer rows."""
    from halite_amd.kernels import ops

    page, table_w = 32, 2
    x, w = rows_of(m, width, m, gpu), rows_of((H + 2 * K) * D, width, H, gpu, 0.2)
    paired = ops.tile_weight(ops.pair_rows_for_rotation(w, D))
    angles = torch.rand((64, D // 2), generator=torch.Generator().manual_seed(5)) * 6
    cos, sin = angles.cos().to(gpu), angles.sin().to(gpu)
    positions = torch.arange(m, dtype=torch.int32) * 3
    table = torch.tensor([[3, 1]], dtype=torch.int32).to(gpu)

    def run(chunks):
        kp = torch.zeros((4, K, page, D), dtype=torch.bfloat16, device=gpu)
        vp = torch.zeros((4, K, D, page), dtype=torch.bfloat16, device=gpu)
        out = []
        for a, b in chunks:
            rows = x[a:b].contiguous()
            if normed:
                sums = torch.full((3, 16), 2.0 * width / 3.0, device=gpu)
                rows = ops.NormedRows(rows, sums, 1e-12, torch.ones(width, device=gpu))
            seg = torch.zeros(b - a, dtype=torch.int32, device=gpu)
            out.append(ops.qkv_rope_append(rows, paired, positions[a:b].to(gpu), cos, sin, H, K, D, seg, table, kp, vp, page, False))
        return torch.cat(out), kp, vp

    for got, want in zip(run([(0, m)]), run([(0, 8), (8, m)])):
        # the product is rounded to bf16, rotated and rounded again: a step of each where sums differ in order
        assert bool(((got.double() - want.double()).abs() <= 2.0 ** -6 * want.double().abs() + 2.0 ** -7 * want.double().abs().max()).all())
        assert float((got != want).double().mean()) < 0.02
        assert float(want.abs().sum()) > 0
