"""The vector forms of the norm with two weights, of the latents' norms and of the heads' columns, and the forms for odd
sizes and addresses, against the same in 64 bits."""

import pytest
import torch

from halite_amd.kernels import ops

pytestmark = pytest.mark.gpu
EPS = 1e-6


def rand(*shape, seed):
    return torch.randn(*shape, generator=torch.Generator().manual_seed(seed)).cuda()


def within(got, want, dtype, sums):
    """One rounding to the result's type and those of a sum of ``sums`` squares (halved by the root), a division and two products."""
    limit = ({torch.bfloat16: 2.0**-8, torch.float32: 0.0}[dtype] + (sums / 2 + 6) * 2.0**-24) * want.abs() + 1e-30
    assert bool(((got.double() - want).abs() <= limit).all())


def normed(x, w):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + EPS) * w


# a vector, an odd size, one more vector than a wave's lanes hold, the widest, rows in other places
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("n, d", [(9, 4), (9, 37), (9, 2052), (9, 4096), (9, 4100), (9, 32768), (255, 260), (256, 4096), (300, 2052)])
def test_norm_with_two_weights(n, d, dtype):
    h, w, second = rand(n, d, seed=1), rand(d, seed=2).to(dtype), rand(d, seed=3).to(dtype)
    rows = torch.tensor([8, 0, 3], dtype=torch.int32, device="cuda")
    for at, want_rows in ((None, h), (rows, h[rows.long()])):
        x, y = ops.rmsnorm_exact(h, w, EPS, dtype, rows=at, second=second)
        alone = ops.rmsnorm_exact(h, w, EPS, dtype, rows=at)
        within(x, normed(want_rows.double(), w.double()), dtype, d), within(y, normed(want_rows.double(), second.double()), dtype, d)
        assert torch.equal(x, alone)


# query latents of no vector, one, 256 threads' worth and one more, the most that threads hold, and more; odd columns
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("q_rank, kv_rank, rot, D, odd", [(0, 64, 0, 64, 0), (4, 4, 4, 16, 0), (1024, 192, 64, 256, 0), (1028, 192, 64, 256, 0),
                                                          (4096, 960, 64, 1024, 0), (4100, 64, 8, 128, 0), (96, 64, 8, 1032, 0), (96, 66, 8, 128, 0), (96, 64, 8, 128, 1)])
def test_latents(q_rank, kv_rank, rot, D, odd, dtype):
    n, heads = 5, 2
    a = rand(n, odd + q_rank + kv_rank + rot + 4, seed=4)
    w_q, w_kv = (rand(q_rank, seed=5).to(dtype) if q_rank else None), rand(kv_rank, seed=6).to(dtype)
    packed = torch.full((n, (heads + 2) * D), 7.0, dtype=dtype, device="cuda")
    cq = ops.latent_prep(a, odd, q_rank, odd + q_rank, kv_rank, rot, D, w_q, w_kv, EPS, packed, heads * D)
    x = a.double()[:, odd:]
    if q_rank:
        within(cq, normed(x[:, :q_rank], w_q.double()), dtype, q_rank)
    keys, values = packed[:, heads * D : (heads + 1) * D], packed[:, (heads + 1) * D :]
    assert bool((packed[:, : heads * D] == 7).all())
    assert torch.equal(keys[:, :rot], a[:, odd + q_rank + kv_rank : odd + q_rank + kv_rank + rot].to(dtype))
    within(keys[:, rot : rot + kv_rank], normed(x[:, q_rank : q_rank + kv_rank], w_kv.double()), dtype, kv_rank)
    assert torch.equal(values[:, rot : rot + kv_rank], keys[:, rot : rot + kv_rank])
    assert not bool(values[:, :rot].any()) and not bool(keys[:, rot + kv_rank :].any()) and not bool(values[:, rot + kv_rank :].any())


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("xs, x0, ys, y0, n, z0, n_zero", [(24, 8, 32, 0, 16, 24, 8), (24, 8, 32, 0, 16, 16, 0), (24, 7, 32, 0, 16, 24, 8), (25, 8, 33, 1, 9, 10, 3)])
def test_columns_of_heads(xs, x0, ys, y0, n, z0, n_zero, dtype):
    heads, tokens = 9, 3
    x, y = rand(tokens, heads * xs, seed=7).to(dtype), rand(tokens, heads * ys, seed=8).to(dtype)
    want = y.clone().view(tokens, heads, ys)
    want[:, :, y0 : y0 + n] = x.view(tokens, heads, xs)[:, :, x0 : x0 + n]
    want[:, :, z0 : z0 + n_zero] = 0
    ops.head_cols(x, xs, x0, y, ys, y0, n, heads, zero_from=z0, n_zero=n_zero)
    assert torch.equal(y.view(tokens, heads, ys), want)
