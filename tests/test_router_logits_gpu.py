"""A router's product in parts of K, and choices made from its planes, against float64 and the choices from whole logits."""

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m, n, k, parts", [
    (1, 16, 512, 2), (16, 64, 4096, 8), (17, 33, 1056, 4), (32, 48, 2048, 8), (33, 1, 544, 2), (64, 256, 4096, 8),  # tiles' edges
    (65, 64, 4096, 0), (8, 257, 2048, 0), (8, 16, 480, 0), (8, 16, 2056, 0),  # left to the other products
])
def test_product_in_parts(gpu, m, n, k, parts):
    from halite_amd.kernels import ops

    gen = torch.Generator().manual_seed(m * 1000 + n)
    x = torch.randn((m, k + 8), generator=gen).bfloat16().to(gpu)[:, :k]
    x = x if parts else x.contiguous()  # (the others take whole rows)
    w = torch.randn((n, k), generator=gen).bfloat16().to(gpu)
    z = ops.router_logits(x, w)
    assert isinstance(z, ops.PartialSums) == (parts > 0) and tuple(z.shape) == (m, n)
    got = z
    if parts:
        assert z.planes.shape == (parts, m, n)
        got = z.planes.double().sum(0)
    want = x.double() @ w.double().T
    # a sum of k products with a rounding at every instruction's 32, each of at most 2^-23 of what has been summed in size
    bound = (x.double().abs() @ w.double().abs().T) * (k / 32 + 16) * 2.0 ** -23
    assert bool(((got.double() - want).abs() <= bound).all())


@pytest.mark.parametrize("tokens, experts, top", [(1, 16, 4), (16, 64, 6), (48, 100, 8), (64, 256, 3)])
def test_choice_from_planes(gpu, tokens, experts, top):
    """Planes of halves of whole numbers, so that their sum is exact in any order: the choice is that of the whole logits."""
    from halite_amd.kernels import ops

    gen = torch.Generator().manual_seed(tokens)
    planes = (torch.randint(-64, 65, (8, tokens, experts), generator=gen) / 16.0).to(gpu)
    for count in (1, 3, 8):
        some = planes[:count].contiguous()
        whole = some.sum(0)
        z = ops.PartialSums(some)
        for a, b in zip(ops.moe_route(z, top, normalize=True), ops.moe_route(whole, top, normalize=True)):
            assert torch.equal(a, b)
        if tokens <= ops.ROUTE_SORT_MAX_TOKENS:
            for a, b in list(zip(ops.moe_route_sort(z, top, experts), ops.moe_route_sort(whole, top, experts)))[:4]:
                assert torch.equal(a, b)
    with pytest.raises(ops.KernelError):
        ops.moe_route(ops.PartialSums(torch.zeros((9, tokens, experts), device=gpu)), top)


def test_not_a_number_stays_one(gpu):
    """A row with an infinity of each sign gives no numbers, as a whole product does, and leaves its neighbours' alone."""
    from halite_amd.kernels import ops

    x, w = torch.ones((20, 1024), device=gpu).bfloat16(), torch.ones((16, 1024), device=gpu).bfloat16()
    x[3, 5], x[3, 900] = float("inf"), float("-inf")
    got = ops.router_logits(x, w).planes.sum(0)
    assert bool(got[3].isnan().all()) and bool((got[[0, 1, 2, 4, 19]] == 1024).all())
