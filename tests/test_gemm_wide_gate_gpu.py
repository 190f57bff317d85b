"""The gates of prompts' products in wide tiles over all that a gate can be, its sum given exactly, against 64 bits."""

import pytest
import torch

from halite_amd.kernels import ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("activation, clamp", [("silu", ops.Clamp()), ("gelu_tanh", ops.Clamp()), ("clamped", ops.Clamp(60.0, 1.0, 0.0)), ("clamped", ops.Clamp(7.0, 1.702, 1.0))])
def test_gates_far_from_zero(activation, clamp):
    gen = torch.Generator().manual_seed(1)
    m, n, k = 700, 256, 128
    # (16 bits each, so that two bf16 terms add up to it)
    whole = torch.cat((torch.linspace(-86, 86, 400), torch.logspace(-30, 1.9, 150), -torch.logspace(-30, 1.9, 150))).float()
    high = whole.bfloat16().float()
    low = (whole - high).bfloat16().float()
    gate = high + low
    up = torch.randn(n, generator=gen).bfloat16()
    x, both = torch.zeros(m, k), torch.zeros(2 * n, k)
    x[:, 5], x[:, 70], x[:, 9] = high, low, 1.0
    both[:n, 5], both[:n, 70], both[n:, 9] = 1.0, 1.0, up.float()
    x, both = x.bfloat16().cuda(), both.bfloat16().cuda()
    y = ops.gemm_bf16_wide(x, both[:n], w_up=both[n:], out_dtype=torch.float32, activation=activation, clamp=clamp)
    g, u = gate.double()[:, None], up.double()[None]
    if activation == "clamped":
        g, u = g.clamp(max=clamp.limit), u.clamp(-clamp.limit, clamp.limit) + clamp.up_shift
        z, turns = clamp.alpha * g, 0 if clamp.alpha == 1 else 1
    elif activation == "silu":
        z, turns = g, 0
    else:
        z, turns = 1.5957691216057308 * (g + 0.044715 * g**3), 6
    want = (g * torch.sigmoid(z) * u).cuda()
    # Units of 2^-24: the power of two 2 (the instruction's) and 1, its sum with one 1, the reciprocal 2, two or three products and the sum of up and
    # shift 4; and `turns` roundings of the sigmoid's argument, which its slope brings in as many times as the argument is large
    limit = (10 + turns * z.abs().cuda()) * 2.0**-24 * want.abs() + 2.0**-126 * g.abs().cuda() * u.abs().cuda()
    off = (y.double() - want).abs()
    assert bool((off <= limit).all()), float((off / limit.clamp(min=1e-300)).max())


def test_gates_without_bounds():
    """The largest numbers, and sums that are infinite: what the quotient g / (1 + exp(-g)) makes of them."""
    n, k = 128, 128
    x, both = torch.zeros(300, k), torch.zeros(2 * n, k)
    x[:, 0], x[:, 1] = torch.tensor([3e38, -3e38, -1e30, 1e30, -100.0, 100.0, -87.0, 0.0, -0.0, 1e-38]).repeat(30), 1.0
    both[:n, 0], both[n:, 1] = torch.tensor([1.0, 2.0]).repeat(n // 2), 0.5  # (twice the largest: infinite)
    x, both = x.bfloat16().cuda(), both.bfloat16().cuda()
    g = x[:, :1].float() * both[:n, 0].float()
    assert bool((g == float("inf")).any()) and bool((g == float("-inf")).any())
    for activation, clamp in (("silu", ops.Clamp()), ("clamped", ops.Clamp(float("inf"), 1.702, 0.0))):
        y = ops.gemm_bf16_wide(x, both[:n], w_up=both[n:], out_dtype=torch.float32, activation=activation, clamp=clamp)
        z = g if activation == "silu" else clamp.alpha * g
        want = g / (1 + torch.exp(-z)) * 0.5
        assert torch.equal(torch.isnan(y), torch.isnan(want))
        plain = ~torch.isnan(want)
        # (the argument's rounding, 2^-24 of up to 170, and what lies below 2^-126 of the gate)
        assert torch.allclose(y[plain], want[plain], rtol=2e-5, atol=2e-36)
