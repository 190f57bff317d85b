"""The weighted sum of the experts' results for many rows (four columns a thread) gives the bits that
the kernel for few rows gives."""

import pytest
import torch

from halite_amd.kernels import ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("d", [4, 252, 1024, 1500, 4096])
@pytest.mark.parametrize("top", [1, 3, 4, 5, 8])
@pytest.mark.parametrize("extra, gated, overwrite", [(False, False, False), (True, False, False), (True, True, True), (False, False, True)])
def test_many_rows_as_few(d, top, extra, gated, overwrite):
    gpu, t = torch.device("cuda:0"), 70
    gen = torch.Generator().manual_seed(d + top)
    h, y, w, e, g = (torch.randn(*shape, generator=gen).to(gpu) for shape in ((t, d), (t * top, d), (t, top), (t, d), (t, 1)))
    pick = lambda a, b: dict(extra=e[a:b] if extra else None, extra_gate=g[a:b] if gated else None, overwrite=overwrite)  # noqa: E731
    many, few = h.clone(), h.clone()
    ops.moe_combine(many, y, w, **pick(0, t))
    for a in range(0, t, 35):  # below 64 rows: a column a thread
        ops.moe_combine(few[a : a + 35], y[a * top : (a + 35) * top], w[a : a + 35], **pick(a, a + 35))
    assert torch.equal(many, few)
    sums = (w.double()[..., None] * y.double().view(t, top, d)).sum(1)
    if extra:
        sums = sums + e.double() * (torch.sigmoid(g.double()) if gated else 1.0)
    want = sums if overwrite else h.double() + sums
    limit = (top + 4) * 2.0**-23 * ((w.abs().double()[..., None] * y.abs().double().view(t, top, d)).sum(1) + e.abs().double() + h.abs().double())
    assert bool(((many.double() - want).abs() <= limit).all())
