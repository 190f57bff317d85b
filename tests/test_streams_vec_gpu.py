"""The pass over copies of the stream in rows of whole groups of four: few and many rows, widths around
its groups of 256 elements and its widest row, against the same sums in 64 bits."""

import pytest
import torch

from halite_amd.kernels import ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("copies, width", [(1, 4), (2, 256), (2, 4096), (2, 4100), (3, 260), (3, 8192), (5, 1028), (8, 4096), (8, 8192)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_few_and_many_rows(copies, width, dtype):
    n, mult, eps = 513, 0.5, 1e-6
    gen = torch.Generator().manual_seed(copies * width)
    x, y = torch.randn(copies, n, width, generator=gen).cuda(), torch.randn(n, width, generator=gen).cuda()
    mix, out, inw = (torch.randn(*shape, generator=gen).cuda() for shape in ((copies, copies), (copies,), (copies,)))
    weight = torch.randn(width, generator=gen).to(dtype).cuda()
    before = x.clone()

    # the steps in 64 bits, and beside each value the sum of its terms' sizes
    new = torch.einsum("sd,stw->dtw", mix.double(), x.double()) + mult * out.double()[:, None, None] * y.double()
    new_size = torch.einsum("sd,stw->dtw", mix.double().abs(), x.double().abs()) + mult * out.double().abs()[:, None, None] * y.double().abs()
    u, u_size = torch.einsum("s,stw->tw", inw.double(), new), torch.einsum("s,stw->tw", inw.double().abs(), new_size)
    norm = (u.square().mean(1, keepdim=True) + eps).sqrt()
    want = u / norm * (1.0 + weight.double())

    args = dict(mix=mix, out=out, mult=mult, read=True, inw=inw, norm_weight=weight, offset=1.0, eps=eps, dtype=dtype)
    got = ops.streams_step(x, y=y, **args).double()
    bit = 2.0**-24
    assert bool(((x.double() - new).abs() <= (copies + 2) * bit * new_size).all())
    u_err = (2 * copies + 3) * bit * u_size
    # the squares: four, six steps over a wave and 32 groups one on the other, and a few operations more
    scale_err = u_err.square().mean(1, keepdim=True).sqrt() / norm + 50 * bit
    bound = u_err / norm * (1.0 + weight.double()).abs() + want.abs() * scale_err
    bound += (2.0**-8 if dtype == torch.bfloat16 else 0.0) * (want.abs() + bound)
    assert bool(((got - want).abs() <= bound).all())

    # few rows: another split of the row, the same bits
    few = before[:, :48].contiguous()
    assert torch.equal(ops.streams_step(few, y=y[:48].contiguous(), **args).double(), got[:48])
    assert torch.equal(few, x[:, :48])
    # chosen rows, only read, into columns of wider rows
    rows = torch.tensor([512, 0, 77], dtype=torch.int32, device="cuda")
    wide = torch.zeros(3, width + 8, dtype=torch.float32, device="cuda")
    ops.streams_step(x, read=True, rows=rows, result=wide[:, 4 : 4 + width])
    plain, size = x[:, rows.long()].double().sum(0), x[:, rows.long()].double().abs().sum(0)
    assert bool(((wide[:, 4 : 4 + width].double() - plain).abs() <= copies * bit * size).all())
    assert not wide[:, :4].any() and not wide[:, 4 + width :].any()
