"""Plans that cut decode tokens' key ranges into more, shorter pieces (as an engine's do): every key once, within the room of a
recorded step, and the same attention as from the longer pieces."""

import numpy as np
import pytest
import torch

from halite_amd.kernels import attention as attn_kernels
from halite_amd.kernels.attention import fix_room_for_decode, pieces_per_tile, plan_items


def ones(n):
    return np.ones(n, dtype=np.int32)


def test_where_shorter_pieces_are_taken():
    spread = lambda n, kv, group, heads: plan_items(ones(n), np.array(kv, dtype=np.int32), group, heads, 0, spread=True)
    # the merge kernel's pieces: four blocks of 32 keys each, one a wave, as many as the room has
    plan = spread(1, [512], 4, 8)
    assert plan.merges.tolist() == [[0, 0, 0, 4, 1, 0, 1, 0]]
    assert plan.items[:, 2:4].tolist() == [[32 * i, 32 * i + 32] for i in range(16)]
    assert spread(1, [255], 4, 8).n_items == 4 and spread(1, [256], 4, 8).n_items == 8
    assert spread(1, [100000], 4, 8).n_items == 4 * 32
    # pieces that the kernel merges: from 1,024 keys on, at most the room's
    assert spread(4, [1023] * 4, 4, 8).n_items == 4 * 4 * 2
    plan = spread(4, [1024] * 4, 4, 8)
    assert plan.n_merges == 0 and plan.n_items == 4 * 4 * 8 and (plan.items[:, 9] == 8).all()
    # a room of one piece, and plans that do not spread, as ever
    assert spread(64, [5000] * 64, 4, 8).n_items == 64 * 4
    assert plan_items(ones(1), np.array([512]), 4, 8, 0).n_items == 4


@pytest.mark.parametrize("head_dim, first", [(64, 512), (112, 512), (128, 384), (256, 384)])
def test_two_pieces_are_never_cut(head_dim, first):
    """What the merge kernel's launch and a second piece's start cost is more than half of so short a walk."""
    assert attn_kernels.spread_from(head_dim) == first
    for n, kv_heads in ((1, 8), (2, 8), (8, 1)):
        count = lambda kv: plan_items(ones(n), np.full(n, kv, dtype=np.int32), 4, kv_heads, 0, spread=first).n_items // 4 // n  # noqa: E731
        assert [count(kv) for kv in (1, 255, 256, 383, first - 1)] == [1] * 5
        assert count(first) == first // 128 and count(first + 127) == first // 128 and count(first + 128) == first // 128 + 1
    # lengths that differ: each by its own
    plan = plan_items(ones(2), np.array([first - 1, first], dtype=np.int32), 4, 8, 0, spread=first)
    assert plan.merges[:, 0].tolist() == [1] and plan.n_items == 4 * (1 + first // 128)
    # inside the kernel as without a line of its own
    for kv in (1023, 1024, 3000):
        a, b = (plan_items(ones(4), np.full(4, kv, dtype=np.int32), 4, 8, 0, spread=s) for s in (first, True))
        assert np.array_equal(a.items, b.items) and a.n_merges == b.n_merges == 0


def test_the_engine_asks_for_that_line(monkeypatch):
    from halite_amd.engine import batch

    asked = []
    monkeypatch.setattr(attn_kernels, "rows_per_big_item", lambda *a: 64)
    monkeypatch.setattr(attn_kernels, "long_items_pay", lambda *a: True)
    monkeypatch.setattr(attn_kernels, "plan_items", lambda *a, spread, **k: asked.append(spread) or plan_items(*a, spread=spread, **k))
    for head_dim in (64, 128, 256):
        ctx = object.__new__(batch.StepContext)
        ctx._plan_host, ctx._dev, ctx.static, ctx.seg_q_len_host, ctx.seg_kv_len_host = {}, None, None, ones(1), np.array([300], np.int32)
        ctx.cache = type("Cache", (), {"groups": [type("Group", (), {"need": object()})]})
        ctx._packer = type("Packer", (), {"add": lambda *a: None})()
        ctx.plan_attention(0, 32, 8, 0, head_dim)
    assert asked == [512, 384, 384]


def test_random_decode_steps_are_covered_and_fit_the_recorded_room():
    rng = np.random.default_rng(11)
    for case in range(300):
        n = int(rng.integers(1, 40))
        group, kv_heads = int(rng.choice([1, 2, 4, 16, 20, 32])), int(rng.choice([1, 2, 8]))
        window = int(rng.choice([0, 0, 37, 1500]))
        kv_len = rng.integers(1, int(rng.choice([300, 2000, 200000])), n).astype(np.int32)
        plan = plan_items(ones(n), kv_len, group, kv_heads, window, 64, spread=True)
        tiles, slots = {}, {}
        for run in plan.items.reshape(-1, 4, plan.items.shape[1]):
            assert len(set(map(tuple, run[:, [0, 1, 4, 5, 6, 7, 8, 9]].tolist()))) == 1
            seg, row, slot, first, count = run[0, [0, 1, 4, 8, 9]].tolist()
            assert run[0, 2] < run[0, 3] and (run[0, 5:8] == [seg, 1, kv_len[seg]]).all()
            tiles.setdefault((seg, row), []).extend((b, e) for b, e in run[:, 2:4].tolist() if e > b)
            slots.setdefault((seg, row), []).append((slot, first, count))
            assert (run[run[:, 3] <= run[:, 2], 2:4] == run[0, 2]).all()  # an empty quarter: the piece's first key twice
        assert sorted(tiles) == [(s, r) for s in range(n) for r in range(0, group, 16)]
        used = []
        for (seg, row), ranges in tiles.items():
            ranges.sort()
            assert ranges[0][0] == (max(0, kv_len[seg] - window) if window else 0) and ranges[-1][1] == kv_len[seg]
            assert all(a[1] == b[0] and a[1] % 32 == 0 for a, b in zip(ranges, ranges[1:]))
            mine = sorted(s for s, _, _ in slots[seg, row])
            entry = [m for m in plan.merges.tolist() if m[:2] == [seg, row]]
            if len(mine) == 1:
                assert mine == [-1] and not entry
                continue
            assert mine == list(range(mine[0], mine[0] + len(mine)))
            used += mine
            if plan.merged_in_kernel:
                assert not entry and set(slots[seg, row]) == {(s, mine[0], len(mine)) for s in mine}
            else:
                assert entry == [[seg, row, mine[0], len(mine), 1, seg, 1, 0]] and all(s[1:] == (0, 0) for s in slots[seg, row])
        assert sorted(used) == list(range(plan.n_partials))
        first = plan_items(ones(n), ones(n), group, kv_heads, window, spread=True)
        fix_room_for_decode(first, n, group, kv_heads)
        assert plan.n_items <= first.cap_items and plan.n_merges <= first.cap_merges and plan.n_partials <= first.cap_partials
        assert plan.max_parts <= pieces_per_tile(n * -(-group // 16), kv_heads)
        if plan.n_partials:
            assert plan.merged_in_kernel == first.merged_in_kernel and (plan.n_merges > 0) == (first.cap_merges > 0)


@pytest.mark.gpu
@pytest.mark.parametrize("K, G, D, lens, window, keep", [
    (8, 4, 128, [256], 0, 0), (8, 4, 128, [511, 2000], 0, 0),  # the merge kernel
    (8, 4, 128, [1024, 1500, 40, 2047], 0, 0), (8, 4, 128, [1024, 1500, 40, 2047], 1100, 0),  # in the kernel
    (1, 32, 256, [700, 1999, 130], 0, 0), (2, 3, 64, [3000, 260], 0, 0), (2, 3, 64, [3000, 1200], 700, 64),
])
def test_shorter_pieces_give_the_same_attention(gpu, K, G, D, lens, window, keep):
    from halite_amd.kernels import ops

    page, n = 64, len(lens)
    gen = torch.Generator().manual_seed(D + n)
    need = [-(-x // page) for x in lens]
    k = torch.randn((sum(need), K, page, D), generator=gen).bfloat16().to(gpu)
    v = torch.randn((sum(need), K, D, page), generator=gen).bfloat16().to(gpu)
    table = torch.full((n, max(need)), -1, dtype=torch.int32)
    order, at = torch.randperm(sum(need), generator=gen).to(torch.int32), 0
    for i, m in enumerate(need):
        table[i, :m] = order[at : at + m]
        at += m
    q = torch.randn((n, K * G * D), generator=gen).bfloat16().to(gpu)
    kv_len = np.array(lens, dtype=np.int32)
    dev = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(gpu)

    class Ctx:
        n_tokens, seg_q_start, seg_q_len, seg_kv_len = n, dev(np.arange(n, dtype=np.int32)), dev(ones(n)), dev(kv_len)

    class Group:
        block_table = table.to(gpu)

    class KV:
        tiled = True

    KV.k, KV.v = k, v
    rule = ops.ScoreRule(keep=keep) if keep else None
    got = []
    for spread in (False, True):
        plan = plan_items(ones(n), kv_len, G, K, window, attn_kernels.rows_per_big_item(D), 0, keep, spread=spread)
        got.append((plan.n_items, attn_kernels.attention_mfma(q, K * G * D, attn_kernels.upload_plan(plan, gpu), Ctx, Group, KV, K * G,
                                                              D ** -0.5, window, rule).double()))
    (few, want), (many, out) = got
    assert many > few
    # probabilities are rounded to bf16 relative to a piece's own maximum (2^-9 of each, once a side), and the result once a side
    bound = 2 * 2.0 ** -9 * float(v.double().abs().max()) + 2 * 2.0 ** -9 * want.abs()
    assert bool(((out - want).abs() <= bound).all())
    assert attn_kernels.counters_idle(gpu)
