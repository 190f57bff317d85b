"""The streaming product of 17 to 64 rows: rows and columns around its tiles, K around its turns through the buffers
(three and six) and in parts, the gated form in both tile widths, rows that lie apart; and the kernels that add up its
planes, against the same kernels on the sum."""

import pytest
import torch

from halite_amd.kernels import ops

pytestmark = pytest.mark.gpu


def rand(gpu, *shape, seed=0, scale=1.0):
    return (scale * torch.randn(*shape, generator=torch.Generator().manual_seed(seed))).to(gpu)


def close(y, want, k):
    """float32 sums of ``k`` exact products of bf16 numbers, rounded to bf16 at most: half a unit in the last
    place (a significand of 8 bits: 2^-8 of the number) plus k roundings of 2^-24 of numbers of the sums' size."""
    err, scale = float((y.double() - want).abs().max()), float(want.abs().max())
    assert err <= (2.0**-8 if y.dtype == torch.bfloat16 else 0.0) * scale + 1e-6 * max(1.0, k / 1024) ** 0.5 * scale, (err, scale)


@pytest.mark.parametrize("m", [17, 32, 33, 64])
@pytest.mark.parametrize("n,k", [(16384, 256), (10244, 320), (20544, 384), (33000, 448), (16384, 1152)])
def test_one_part(gpu, m, n, k):
    x, w = rand(gpu, m, k + 8, seed=1).bfloat16()[:, :k], rand(gpu, n, k, seed=2, scale=0.05).bfloat16()
    parts = ops.stream_parts(x, w, n)
    assert parts == 1
    want = x.double() @ w.double().t()
    for dtype in (torch.bfloat16, torch.float32):
        close(ops.gemm_bf16_stream(x, w, parts, out_dtype=dtype), want, k)


@pytest.mark.parametrize("m", [17, 32, 33, 50, 64])
@pytest.mark.parametrize("n,k,parts", [(4096, 4096, 4), (6144, 1024, 2), (6144, 4096, 5), (4096, 14336, 4), (2048, 3200, 8), (3000, 2112, 5), (6144, 832, 2)])
def test_planes(gpu, m, n, k, parts):
    x, w = rand(gpu, m, k, seed=3).bfloat16(), rand(gpu, n, k, seed=4, scale=0.05).bfloat16()
    assert ops.stream_parts(x, w, n, may_part=True) == parts
    got = ops.gemm_bf16_stream(x, w, parts)
    want = x.double() @ w.double().t()
    assert isinstance(got, ops.PartialSums) and got.shape == (m, n)
    close(got.planes.sum(0), want, k)
    close(got.materialize(torch.float32), want, k)
    close(got.materialize(torch.bfloat16), want, k)


@pytest.mark.parametrize("m", [17, 48, 64])
@pytest.mark.parametrize("f,k", [(14336, 512), (8192, 320), (11008, 256), (5500, 704)])  # tiles of 64 + 64 and of 32 + 32 rows
@pytest.mark.parametrize("activation", ["silu", "clamped"])
def test_gated(gpu, m, f, k, activation):
    x, w = rand(gpu, m, k, seed=5).bfloat16(), rand(gpu, 2 * f, k, seed=6, scale=0.1).bfloat16()
    assert ops.stream_parts(x, w, f, gated=True) == 1
    clamp = ops.Clamp(1.5, 1.7, 1.0) if activation == "clamped" else ops.Clamp()
    y = ops.gemm_bf16_stream(x, w[:f], 1, w_up=w[f:], activation=activation, clamp=clamp)
    g, u = x.double() @ w[:f].double().t(), x.double() @ w[f:].double().t()
    if activation == "clamped":
        g, u = g.clamp(max=1.5), u.clamp(-1.5, 1.5)
        want = g * torch.sigmoid(1.7 * g) * (u + 1.0)
    else:
        want = g * torch.sigmoid(g) * u
    assert float((y.double() - want).abs().max()) <= (2.0**-8 + 1e-5) * float(want.abs().max())


@pytest.mark.parametrize("n,k,rows", [(10304, 3072, 8), (16380, 2048, 12), (12801, 3072, 16), (4096, 3072, 16)])
def test_bare_products_of_few_rows(gpu, n, k, rows):
    """A product that folds nothing in leaves the small-batch kernel above ``rows`` rows, where one part fills the chip and columns are
    whole vectors."""
    w = rand(gpu, n, k, seed=14, scale=0.05).bfloat16()
    tiled = ops.tile_weight(w)
    for m in (1, rows, min(rows + 1, 16), 16):
        x = rand(gpu, m, k, seed=m).bfloat16()
        got = ops.linear(x, w, out_dtype=torch.float32, tiled=tiled)
        close(got, x.double() @ w.double().t(), k)
        same = ops.gemm_bf16_stream(x, w, 1, out_dtype=torch.float32) if m > rows else ops.gemm_bf16_skinny(x, tiled, out_dtype=torch.float32, tiled_shape=(n, k))
        assert torch.equal(got, same)
        assert torch.equal(ops.linear(x, w, tiled=tiled), got.bfloat16())


def test_what_it_does_not_take(gpu):
    w = torch.zeros((4096, 4096), dtype=torch.bfloat16, device=gpu)
    x = lambda m, k=4096: torch.zeros((m, k), dtype=torch.bfloat16, device=gpu)  # noqa: E731
    assert ops.stream_parts(x(17), w, 4096, may_part=True) == 4
    assert not ops.stream_parts(x(16), w, 4096, may_part=True) and not ops.stream_parts(x(65), w, 4096, may_part=True)
    assert not ops.stream_parts(x(17), w, 4096)  # (one part would leave the chip idle)
    assert not ops.stream_parts(x(17, 4097)[:, 1:], w, 4096, may_part=True)  # off 16 bytes
    assert not ops.stream_parts(x(17, 4000), w[:, :4000], 4096, may_part=True)  # K of half a step
    assert not ops.stream_parts(x(17).float(), w, 4096, may_part=True)


@pytest.mark.parametrize("rows,d,n_planes", [(17, 4096, 4), (64, 3072, 5), (33, 8192, 2), (20, 260, 9), (17, 16388, 2), (17, 32768, 2), (17, 32772, 2)])
def test_the_norm_adds_up_planes(gpu, rows, d, n_planes):
    planes = ops.PartialSums(rand(gpu, n_planes, rows, d, seed=7))
    h, w = rand(gpu, rows, d, seed=8), rand(gpu, d, seed=9).bfloat16()
    h2 = h.clone()
    x = ops.rmsnorm(h, w, 1e-5, torch.bfloat16, delta=planes)
    y = ops.rmsnorm(h2, w, 1e-5, torch.bfloat16, delta=planes.materialize(torch.bfloat16))
    assert torch.equal(x, y) and torch.equal(h, h2)
    some = torch.tensor([rows - 1, 3, 3], dtype=torch.int32, device=gpu)  # rows alone leave the stream as it is
    x = ops.rmsnorm(h, w, 1e-5, torch.bfloat16, delta=planes, rows=some)
    assert torch.equal(h, h2)
    assert torch.equal(x, ops.rmsnorm(h2, w, 1e-5, torch.bfloat16, delta=planes.materialize(torch.bfloat16), rows=some))


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("off_h, off_w", [(0, 1), (0, 2), (1, 0), (3, 3)])
def test_a_norm_off_the_kernels_places(gpu, off_h, off_w, dtype):
    """Weights and streams that begin inside a vector: taken as with a delta in one piece."""
    rows, d = 18, 512
    planes = ops.PartialSums(rand(gpu, 3, rows, d, seed=13))
    w = rand(gpu, d + off_w, seed=14).to(dtype)[off_w:]
    h, h2 = (rand(gpu, rows * d + off_h, seed=15)[off_h:].view(rows, d) for _ in range(2))
    x = ops.rmsnorm(h, w, 1e-5, torch.bfloat16, delta=planes)
    y = ops.rmsnorm(h2, w, 1e-5, torch.bfloat16, delta=planes.materialize(torch.bfloat16))
    assert torch.equal(x, y) and torch.equal(h, h2)


@pytest.mark.parametrize("off", [0, 1])  # (tables that begin inside a vector)
@pytest.mark.parametrize("H,K,D,page,tiled", [(32, 8, 128, 64, True), (24, 8, 128, 64, True), (6, 2, 48, 16, False), (4, 4, 16, 8, False)])
def test_the_rotation_adds_up_planes(gpu, H, K, D, page, tiled, off):
    n, segs, n_planes = 37, 5, 3
    planes = ops.PartialSums(rand(gpu, n_planes, n, (H + 2 * K) * D, seed=10))
    i32 = lambda t: t.to(torch.int32).to(gpu)  # noqa: E731
    seg, pos = i32(torch.arange(n) % segs), i32(torch.arange(n) // segs * 3 + 50)
    table = i32(torch.randperm(40, generator=torch.Generator().manual_seed(11))[: segs * 8].view(segs, 8))
    angles = rand(gpu, 8 * page if 8 * page > 80 else 80, D // 2, seed=12)
    pages = lambda *shape: torch.zeros(shape, dtype=torch.bfloat16, device=gpu)  # noqa: E731
    pos = pos % (8 * page)
    k1, v1, k2, v2 = pages(40, K, page, D), pages(40, K, D, page), pages(40, K, page, D), pages(40, K, D, page)
    cos, sin = (torch.cat((t.new_zeros(off), t.flatten()))[off:].view(t.shape) for t in (torch.cos(angles), torch.sin(angles)))
    q = ops.rope_append_sums(planes, pos, cos, sin, H, K, D, seg, table, k1, v1, page, tiled)
    rows = planes.materialize(torch.bfloat16)
    ops.rope_append(rows, pos, cos, sin, H, K, D, D, False, token_seg=seg, block_table=table, k_pages=k2, v_pages=v2, page_size=page, tiled=tiled)
    # (a turned pair's two products may be added with one rounding or with two: a step of bf16 where that decides, or of float32
    # where the two nearly cancel)
    for got, want in ((q, rows[:, : H * D]), (k1, k2)):
        assert torch.allclose(got.float(), want.float(), rtol=2.0**-7, atol=1e-6) and float((got != want).float().mean()) < 1e-3
    assert torch.equal(v1, v2)


@pytest.mark.parametrize("m", [17, 48, 64])
@pytest.mark.parametrize("n,k,gated", [(20544, 4096, False), (32001 // 4 * 4, 4160, False), (20484, 4224, False), (11008, 4096, True), (12288, 4160, True),
                                       (12292, 4096, True), (20544, 4032, False)])
def test_long_rows_through_six_buffers(gpu, m, n, k, gated):
    """One workgroup a compute unit and 64 steps of K or more (4,032 and 12,292 gated: the three buffers still); steps that
    do not fill the last turn through the buffers."""
    x, w = rand(gpu, m, k, seed=21).bfloat16(), rand(gpu, n, k, seed=22, scale=0.05).bfloat16()
    up = rand(gpu, n, k, seed=23, scale=0.05).bfloat16() if gated else None
    assert ops.stream_parts(x, w, n, gated=gated) == 1
    y = ops.gemm_bf16_stream(x, w, 1, w_up=up, out_dtype=torch.float32 if not gated else torch.bfloat16)
    want, size = x.double() @ w.double().t(), x.double().abs() @ w.double().abs().t()
    steps = (k / 32 + 8) * 2.0 ** -23  # a rounding of each partial sum
    if gated:
        u, u_size = x.double() @ up.double().t(), x.double().abs() @ up.double().abs().t()
        s = want * torch.sigmoid(want)
        bound = (1.1 * size * u.abs() + s.abs() * u_size) * steps + (s * u).abs() * 2.0 ** -7.9 + 1e-6
        want = s * u
    else:
        bound = size * steps
    assert bool(((y.double() - want).abs() <= bound).all())
