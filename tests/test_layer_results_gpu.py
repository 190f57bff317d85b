"""Norms that add what a layer left to the stream first, against the passes one by one: the same bits of the stream, and rows of its norm."""

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("t, d, top, beside, extra", [
    (1, 4, 1, False, None), (8, 4096, 6, False, "plain"), (17, 1028, 5, True, "plain"), (64, 2048, 4, True, "gated"), (300, 4100, 3, True, None),
    (3, 16384, 8, True, "gated"), (5, 1030, 2, True, "plain"), (2, 16388, 2, False, None),  # the last two: one by one
])
@pytest.mark.parametrize("pair", [False, True])
def test_as_one_by_one(gpu, t, d, top, beside, extra, pair):
    from halite_amd.kernels import ops

    gen = torch.Generator().manual_seed(t + d)
    rnd = lambda *s: torch.randn(s, generator=gen).to(gpu)
    h0 = rnd(t, d)
    wide = rnd(t, 3)
    e = ops.ExpertSum(rnd(t * top, d), torch.rand((t, top), generator=gen).to(gpu), None if extra is None else rnd(t, d),
                      wide[:, 2:] if extra == "gated" else None)
    left = ops.LayerResults(rnd(t, d) if beside else None, e)
    w = rnd(d).bfloat16()
    second = rnd(d).bfloat16() if pair else None
    ha, hb = h0.clone(), h0.clone()
    left.add_to(ha)
    want = ops.rmsnorm_exact(ha, w, 1e-5, torch.float32, second=second)
    got = ops.rmsnorm_exact(hb, w, 1e-5, torch.float32, second=second, added=left)
    # the same sums in the same order; a sum's multiply-adds may be fused in one and not in the other
    size = h0.abs() + (left.beside.abs() if beside else 0) + (e.y.view(t, top, d).abs() * e.wgt[:, :, None]).sum(1) + (0 if extra is None else e.extra.abs())
    assert bool(((ha - hb).abs() <= size * (top + 4) * 2.0 ** -24).all())
    for a, b in zip(want if pair else (want,), got if pair else (got,)):
        assert bool(((a - b).abs() <= 2.0 ** -18 * (a.abs() + 1e-3) * (top + 4) + size * w.float().abs().max() * 2.0 ** -18).all())
    # chosen rows: the same rows, and the stream is as it was (or has what was to be added)
    rows = torch.tensor([t - 1, 0, t // 2], dtype=torch.int32, device=gpu)
    hc = h0.clone()
    some = ops.rmsnorm_exact(hc, w, 1e-5, torch.float32, rows=rows, second=second, added=left)
    for a, b in zip(some if pair else (some,), got if pair else (got,)):
        assert torch.equal(a, b[rows.long()])
    assert torch.equal(hc, h0) or torch.equal(hc, hb)


def test_what_is_refused(gpu):
    from halite_amd.kernels import ops

    h, w = torch.zeros((3, 16), device=gpu), torch.ones(16, device=gpu)
    good = lambda: ops.ExpertSum(torch.zeros((6, 16), device=gpu), torch.zeros((3, 2), device=gpu))
    ops.rmsnorm_exact(h, w, 1e-5, torch.float32, added=ops.LayerResults(None, good()))
    for bad in (ops.LayerResults(torch.zeros((2, 16), device=gpu), good()),
                ops.LayerResults(None, ops.ExpertSum(torch.zeros((5, 16), device=gpu), torch.zeros((3, 2), device=gpu))),
                ops.LayerResults(None, ops.ExpertSum(torch.zeros((6, 16), device=gpu), torch.zeros((3, 2), device=gpu), None,
                                                     torch.zeros((3, 1), device=gpu)))):
        with pytest.raises(ops.KernelError):
            ops.rmsnorm_exact(h, w, 1e-5, torch.float32, added=bad)
