"""The step of a stream in several copies with a result that it adds up itself (planes of a product, experts' rows), against the
same step with the result added up before."""

import pytest
import torch

pytestmark = pytest.mark.gpu


def numbers(gen, *shape):
    return torch.randn(shape, generator=gen)


@pytest.mark.parametrize("what", ["planes", "experts", "beside", "gated"])
@pytest.mark.parametrize("copies, t, w, terms", [
    (1, 3, 4, 1), (2, 48, 2048, 4), (2, 5, 4100, 8), (3, 17, 1028, 5), (4, 64, 8192, 3), (2, 640, 4096, 4),  # the last: two groups a thread
    (2, 9, 1026, 4), (5, 6, 256, 2), (2, 2, 8196, 3),  # added up before: no whole groups, too many copies, too wide
])
def test_as_added_up_before(gpu, what, copies, t, w, terms):
    from halite_amd.kernels import ops

    gen = torch.Generator().manual_seed(copies * 1000 + t)
    x0 = numbers(gen, copies, t, w).to(gpu)
    mix, out, inw = (numbers(gen, *s).to(gpu) for s in ((copies, copies), (copies,), (copies,)))
    weight = numbers(gen, w).bfloat16().to(gpu)
    if what == "planes":
        y = ops.PartialSums(numbers(gen, terms, t, w).to(gpu))
        whole, size = y.planes.double().sum(0), y.planes.double().abs().sum(0)
    else:
        extra = numbers(gen, t, w).to(gpu) if what != "experts" else None
        wide = numbers(gen, t, 3).to(gpu)
        gate = wide[:, 1:2] if what == "gated" else None
        y = ops.ExpertSum(numbers(gen, t * terms, w).to(gpu), torch.rand((t, terms), generator=gen).to(gpu), extra, gate)
        rows = y.y.view(t, terms, w).double() * y.wgt.double()[:, :, None]
        beside = 0.0 if extra is None else extra.double() * (1.0 if gate is None else torch.sigmoid(gate.double()))
        whole, size = rows.sum(1) + beside, rows.abs().sum(1) + (0.0 if extra is None else beside.abs())
    args = dict(mix=mix, out=out, mult=0.5, read=True, inw=inw, norm_weight=weight, offset=1.0, eps=1e-5)
    before = y.materialize(torch.float32) if what == "planes" else y.materialize()
    # a sum of so many float32 terms: a rounding of each partial sum (and of the sigmoid and its product)
    assert bool(((before.double() - whole).abs() <= size * (terms + 4) * 2.0 ** -23).all())
    xa, xb = x0.clone(), x0.clone()
    a = ops.streams_step(xa, y=before, dtype=torch.float32, **args)
    b = ops.streams_step(xb, y=y, dtype=torch.float32, **args)
    moved = size[None] * out.double().abs()[:, None, None] * 0.5 * (terms + 4) * 2.0 ** -22
    large = torch.einsum("std,so->otd", x0.double().abs().cpu(), mix.double().abs().cpu()).to(gpu) * (copies + 2) * 2.0 ** -23
    assert bool(((xa.double() - xb.double()).abs() <= moved + large).all())
    # the norm: a relative change of the row and of its size
    u = torch.einsum("std,s->td", xa.double().cpu(), inw.double().cpu()).to(gpu)
    change = ((moved + large + xa.double().abs() * 2.0 ** -22) * inw.double().abs()[:, None, None]).sum(0)
    scale = 1.0 / torch.sqrt((u ** 2).mean(1, keepdim=True) + 1e-5)
    factor = (1.0 + weight.double()).abs()
    bound = factor * scale * (change + u.abs() * ((change ** 2).mean(1, keepdim=True).sqrt() * scale + 2.0 ** -18)) + 1e-7
    assert bool(((a.double() - b.double()).abs() <= bound).all())
    # nothing read, and read as it is into wider rows
    xc, xd = x0.clone(), x0.clone()
    ops.streams_step(xc, y=y, mix=mix, out=out, mult=0.5)
    assert torch.equal(xc, xb)
    wide_rows = torch.zeros((t, w + 8), device=gpu)
    ops.streams_step(xd, y=y, mix=mix, out=out, mult=0.5, read=True, result=wide_rows[:, 3 : w + 3])  # (a place that the vector kernel does not take)
    aligned = torch.zeros((t, w + 8), device=gpu)
    xe = x0.clone()
    ops.streams_step(xe, y=y, mix=mix, out=out, mult=0.5, read=True, result=aligned[:, 4 : w + 4])
    want = xe.double().sum(0)
    slack = xe.double().abs().sum(0) * (copies + 1) * 2.0 ** -22 + (moved + large).sum(0)
    for got in (wide_rows[:, 3 : w + 3], aligned[:, 4 : w + 4]):
        assert bool(((got.double() - want).abs() <= slack).all())
    assert float(aligned[:, :4].abs().max()) == 0 and float(aligned[:, w + 4 :].abs().max()) == 0


def test_what_is_refused(gpu):
    from halite_amd.kernels import ops

    x = torch.zeros((2, 3, 16), device=gpu)
    args = dict(mix=torch.eye(2, device=gpu), out=torch.ones(2, device=gpu))
    for bad in (ops.PartialSums(torch.zeros((2, 4, 16), device=gpu)), ops.PartialSums(torch.zeros((2, 3, 16), device=gpu).bfloat16()),
                ops.ExpertSum(torch.zeros((7, 16), device=gpu), torch.zeros((3, 2), device=gpu)),
                ops.ExpertSum(torch.zeros((6, 16), device=gpu), torch.zeros((3, 2), device=gpu), None, torch.zeros((3, 1), device=gpu))):
        with pytest.raises(ops.KernelError):
            ops.streams_step(x, y=bad, **args)
