"""Element-wise passes of prompts in vectors and runs: the convolution in runs of eight tokens, heads' gates four columns a thread, rows
of zeros in several arrays."""

import pytest
import torch

from halite_amd.kernels import ops

pytestmark = pytest.mark.gpu


def i32(values):
    return torch.tensor(values, dtype=torch.int32, device="cuda")


# lengths of segments around a run and the taps, so that runs begin inside a segment, at its start and a few tokens behind; the last run
# cut; channels that end inside a workgroup; and (the second place of `apart`) inputs off a vector, which go a token a thread
@pytest.mark.parametrize("lengths", [[2051], [1, 2, 3, 4, 5, 900, 1, 1, 7, 8, 9, 1200], [1023, 1025]])
@pytest.mark.parametrize("taps", [2, 3, 4, 5])
@pytest.mark.parametrize("apart", [(8, 0), (8, 1), (0, 0)])
@pytest.mark.parametrize("how", [dict(), dict(bias=True, in_bias=True, silu=True, out=torch.bfloat16)])
def test_convolution_in_runs(lengths, taps, apart, how):
    n, c = sum(lengths), 1028
    gen = torch.Generator().manual_seed(n + taps)
    rand = lambda *shape: torch.randn(*shape, generator=gen).cuda()  # noqa: E731
    u = rand(n, c + apart[0])[:, apart[1] : apart[1] + c]
    w, state = rand(c, taps).bfloat16(), rand(len(lengths) + 1, taps - 1, c)
    bias, in_bias = (rand(c).bfloat16(), rand(c)) if how.get("bias") else (None, None)
    slots = [len(lengths) - s for s in range(len(lengths))]
    starts = [sum(lengths[:s]) for s in range(len(lengths))]
    of = [s for s, length in enumerate(lengths) for _ in range(length)]
    got = ops.short_conv(u, w, bias, state, i32(of), i32(starts), i32([slots[s] for s in of]), how.get("out", torch.float32),
                         silu=bool(how.get("silu")), in_bias=in_bias)
    for s, (t0, length) in enumerate(zip(starts, lengths)):
        x = u[t0 : t0 + length].double() + (in_bias.double() if in_bias is not None else 0.0)
        joined = torch.cat([state[slots[s]].double(), x])
        want = sum(w.double()[:, j] * joined[j : j + length] for j in range(taps)) + (bias.double() if bias is not None else 0.0)
        size = sum(w.double()[:, j].abs() * joined[j : j + length].abs() for j in range(taps)) + 4.0
        if how.get("silu"):
            want = want * torch.sigmoid(want)
        # a rounding a tap, the input's bias and the gate; a bfloat16 result another of 2^-9
        limit = (taps + 6) * 2.0**-24 * size + (2.0**-8 * want.abs() if got.dtype == torch.bfloat16 else 0.0)
        assert bool(((got[t0 : t0 + length].double() - want).abs() <= limit).all())
    # few tokens go a token a thread: the same numbers
    few = min(lengths[0], 40)
    part = ops.short_conv(u[:few], w, bias, state, i32([0] * few), i32([0]), i32([slots[0]] * few), how.get("out", torch.float32),
                          silu=bool(how.get("silu")), in_bias=in_bias)
    assert torch.equal(part, got[:few])


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("rows", [1, 64, 65, 300])
@pytest.mark.parametrize("heads, n, apart", [(3, 4, 4), (32, 128, 128), (5, 64, 80), (20, 100, 100), (3, 6, 8), (4, 64, 66)])  # (the last two: an entry a thread)
def test_heads_gates(dtype, rows, heads, n, apart):
    gen = torch.Generator().manual_seed(rows + heads)
    x, g = torch.randn(rows, heads * apart, generator=gen).cuda().to(dtype), torch.randn(rows, heads, generator=gen).cuda()
    got = ops.head_gate_cols(x, apart, g, n, heads)
    want = (x.view(rows, heads, apart)[:, :, :n].double() * torch.sigmoid(g.double())[:, :, None]).reshape(rows, heads * n)
    assert got.shape == want.shape and bool(((got.double() - want).abs() <= (2.0**-8 if dtype == torch.bfloat16 else 4e-7) * want.abs() + 1e-30).all())


def test_rows_of_zeros():
    shapes = [((5, 64, 64, 64), torch.float32), ((5, 3, 7), torch.float32), ((5, 3), torch.bfloat16), ((5, 6), torch.bfloat16), ((5, 0, 4), torch.float32)]
    tensors = [torch.ones(shape, dtype=dtype, device="cuda") for shape, dtype in shapes * 20]  # (more than one launch takes)
    ops.zero_rows(tensors, 3)
    for t in tensors:
        assert bool((t[3] == 0).all()) and bool((t[:3] == 1).all()) and bool((t[4:] == 1).all())
    with pytest.raises(ops.KernelError):
        ops.zero_rows(tensors, 5)
