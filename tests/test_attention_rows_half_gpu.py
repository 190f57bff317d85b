"""Float32 attention of prompts in workgroups of 64 rows (where those of 128 leave half of the compute units without one): bit for bit what the
larger ones give, whatever the rule, the pages and the places of the range's ends."""

import pytest
import torch

from halite_amd.kernels import ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("H, K, D, before, new, page, window, keep, rule", [
    (32, 8, 128, 0, 512, 64, 0, 0, {}), (32, 8, 128, 0, 33, 16, 0, 0, {}), (32, 8, 128, 3, 257, 16, 0, 0, {}),  # 128 workgroups of 128 rows; one; a range
    (32, 8, 128, 61, 130, 16, 37, 0, {}), (32, 8, 128, 61, 130, 16, 38, 6, {}), (32, 8, 128, 500, 75, 16, 2, 0, {}),  # that ends among four keys
    (32, 8, 120, 70, 61, 6, 0, 0, {}), (16, 2, 64, 9, 200, 10, 45, 0, {}),  # pages of no multiple of four
    (160, 2, 32, 5, 3, 16, 0, 0, {}), (24, 8, 96, 33, 129, 8, 0, 0, dict(softcap=20.0)),  # more heads a key/value head than rows
    (8, 1, 24, 40, 333, 16, 0, 0, dict(sigmoid=True)), (12, 4, 72, 12, 77, 16, 50, 0, dict(bias=True)),
])
def test_as_in_larger_workgroups(gpu, H, K, D, before, new, page, window, keep, rule):
    gen = torch.Generator().manual_seed(D + new)
    rnd = lambda *s: torch.randn(s, generator=gen)  # noqa: E731
    others = [(3, 1021)] * 16
    segs = [(before, new)] + others
    pages = [-(-(b + n) // page) for b, n in segs]
    tables = torch.full((len(segs), max(pages)), -1, dtype=torch.int32)
    order, at = torch.randperm(sum(pages), generator=gen).to(torch.int32), 0
    for i, n in enumerate(pages):
        tables[i, :n] = order[at : at + n]
        at += n
    k, v = rnd(sum(pages), K, page, D), rnd(sum(pages), K, D, page)
    # slots that nothing has been written to, and keys before a window, must not matter
    last = before + new
    if last % page:
        k[int(tables[0, last // page]), :, last % page :] = float("nan")
        v[int(tables[0, last // page]), :, :, last % page :] = float("nan")
    k, v = k.to(gpu), v.to(gpu)
    q = [rnd(n, H * D) for _, n in segs]
    kind = dict(rule)
    if kind.pop("bias", False):
        kind["bias"] = rnd(H, 64).to(gpu)
    how = ops.ScoreRule(keep=keep, **kind)

    def run(which):
        i32 = lambda t: t.to(torch.int32).to(gpu)  # noqa: E731
        out = ops.attention_simple(
            torch.cat([q[i] for i in which]).to(gpu), H * D, i32(torch.cat([torch.arange(segs[i][0], sum(segs[i])) for i in which])),
            i32(torch.cat([torch.full((segs[i][1],), j) for j, i in enumerate(which)])), tables[which].to(gpu), k, v, H, D**-0.5, window,
            max_kv_len=max(sum(segs[i]) for i in which), min_q_len=min(segs[i][1] for i in which), rule=how)
        return out[:new]

    workgroups = lambda which: -(-sum(segs[i][1] for i in which) // max(1, 128 // (H // K))) * K * -(-(H // K) // 128)  # noqa: E731
    most = list(range(len(segs)))
    assert workgroups([0]) <= 128
    alone = run([0])
    assert bool(torch.isfinite(alone).all())
    seen = set()
    for n in range(2, len(segs) + 1):  # each of the larger builds once
        w = most[:n]
        size = "one" if workgroups(w) > 256 else "two" if workgroups(w) > 128 else None
        if size and size not in seen:
            seen.add(size)
            assert torch.equal(alone, run(w)), size
    assert seen


def test_a_hole_in_the_table_shows(gpu):
    H, K, D, page, new = 8, 2, 64, 16, 64
    gen = torch.Generator().manual_seed(1)
    k, v = torch.randn((4, K, page, D), generator=gen).to(gpu), torch.randn((4, K, D, page), generator=gen).to(gpu)
    q = torch.randn((new, H * D), generator=gen).to(gpu)
    table = torch.tensor([[0, 1, -1, 3]], dtype=torch.int32, device=gpu)
    out = ops.attention_simple(q, H * D, torch.arange(new, dtype=torch.int32, device=gpu), torch.zeros(new, dtype=torch.int32, device=gpu), table,
                               k, v, H, D**-0.5, 0, max_kv_len=new, min_q_len=new, rule=None)
    assert bool(torch.isfinite(out[:32]).all()) and bool(torch.isnan(out[32:]).all())
