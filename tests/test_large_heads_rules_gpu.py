"""The attention kernel for long segments at every head size over 128 that it is built for, with every rule
for the scores that it knows, against the same attention in 64 bits; one-tile items beside it."""

import types

import numpy as np
import pytest
import torch

from halite_amd.kernels import attention as attn_kernels
from halite_amd.kernels import ops
from test_kernels_gpu import paged_cache, rnd, to_tiled

SEGS = [(0, 1), (0, 70), (63, 40), (300, 5), (130, 150)]  # tokens before, new tokens
HEADS, KV = 8, 2
N_BIASES = 50


def plain(q, k, v, scale, window, rule):
    """Every token's result in 64 bits, and beside it the sum of its terms without their signs."""
    n, heads, d = q.shape
    q, k, v = q.double(), k.double(), v.double()
    rows, cols = torch.arange(n).unsqueeze(1), torch.arange(n).unsqueeze(0)
    hidden = cols > rows
    if window:
        hidden = hidden | ((cols <= rows - window) & (cols >= rule.keep))
    if rule.chunk:
        hidden = hidden | (cols < rows // rule.chunk * rule.chunk)
    out, size = torch.empty_like(q), torch.empty_like(q)
    for h in range(heads):
        g = h // (heads // k.shape[1])
        s = q[:, h] @ k[:, g].T * scale
        if rule.softcap:
            s = rule.softcap * torch.tanh(s / rule.softcap)
        if rule.bias is not None:
            s = s + rule.bias[h].double().cpu()[(rows - cols).clamp(0, N_BIASES - 1)]
        if rule.sigmoid:
            p = torch.sigmoid(s).masked_fill(hidden, 0.0)
        else:
            s = s.masked_fill(hidden, float("-inf"))
            if rule.sink:
                sink = torch.zeros(n, 1) if rule.sink_values is None else rule.sink_values[h].cpu().expand(n, 1)
                s = torch.cat((s, sink.double()), 1)
            p = torch.softmax(s, 1)[:, :n]
        out[:, h], size[:, h] = p @ v[:, g], p @ v[:, g].abs()
    return out, size


def rule_of(name):
    log2e = 1.4426950408889634
    bias, sinks = rnd(HEADS, N_BIASES, seed=70).cuda(), rnd(HEADS, seed=71).cuda()
    return {
        "none": (0, ops.ScoreRule()),
        "window": (37, ops.ScoreRule()),
        "kept": (37, ops.ScoreRule(keep=20)),
        "chunks": (0, ops.ScoreRule(chunk=48)),
        "sinks": (0, ops.ScoreRule(sink=True, sink_values=sinks, sink_values_log2=sinks * log2e)),
        "bias and sink": (90, ops.ScoreRule(bias=bias, bias_log2=bias * log2e, sink=True)),
        "cap": (0, ops.ScoreRule(softcap=2.0)),
        "sigmoid": (0, ops.ScoreRule(sigmoid=True, bias=bias, bias_log2=bias * log2e)),
    }[name]


@pytest.mark.gpu
@pytest.mark.parametrize("rule_name", ["none", "window", "kept", "chunks", "sinks", "bias and sink", "cap", "sigmoid"])
@pytest.mark.parametrize("D, value_from", [(144, 0), (160, 0), (176, 0), (192, 64), (208, 0), (224, 0), (256, 64)])
def test_rules(D, value_from, rule_name):
    gpu, page = torch.device("cuda:0"), 64
    window, rule = rule_of(rule_name)
    skipped = attn_kernels.skips_leading_zeros(D, value_from) and not rule.keep
    qs, ks, vs, tables, want, size, base = [], [], [], [], [], [], 0
    for i, (before, new) in enumerate(SEGS):
        n = before + new
        q, k, v = (rnd(n, h, D, seed=90 + 3 * i + j).bfloat16().float() for j, h in enumerate((HEADS, KV, KV)))
        v[..., :value_from] = 0
        w, s = plain(q, k, v, D**-0.5, window, rule)
        want.append(w[before:]), size.append(s[before:])
        qs.append(q[before:].reshape(new, -1))
        if skipped:  # what is not to be read shows
            v[..., :value_from] = float("nan")
        kp, vp, table = paged_cache(k, v, page, 30 + i, dtype=torch.bfloat16)
        ks.append(kp), vs.append(vp), tables.append(table + base)
        base += kp.shape[0]
    bt = torch.full((len(SEGS), max(len(t) for t in tables)), -1, dtype=torch.int32)
    for i, t in enumerate(tables):
        bt[i, : len(t)] = t
    k_pages, v_pages = torch.cat(ks), torch.cat(vs)
    tiled = D % 32 == 0
    if tiled:
        k_pages, v_pages = to_tiled(k_pages, v_pages)
    q_len, kv_len = (np.array(a, dtype=np.int32) for a in ([n for _, n in SEGS], [b + n for b, n in SEGS]))
    dev = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(gpu)  # noqa: E731
    starts = np.concatenate(([0], np.cumsum(q_len)[:-1])).astype(np.int32)
    ctx = types.SimpleNamespace(n_tokens=int(q_len.sum()), seg_q_start=dev(starts), seg_q_len=dev(q_len), seg_kv_len=dev(kv_len))
    kv = types.SimpleNamespace(k=k_pages.to(gpu), v=v_pages.to(gpu), tiled=tiled, value_from=value_from)
    want, size = torch.cat(want), torch.cat(size)
    rows_big = attn_kernels.rows_per_big_item(D, 0 if rule.keep else value_from)
    assert rows_big == (16 if D == 256 and rule.keep else 32)
    for rows in sorted({rows_big, attn_kernels.ROWS_PER_ITEM}):
        plan = attn_kernels.plan_items(q_len, kv_len, HEADS // KV, KV, window, rows, rule.chunk, rule.keep)
        assert (plan.n_big > 0) == (rows > 16)
        got = attn_kernels.attention_mfma(torch.cat(qs).bfloat16().to(gpu), HEADS * D, attn_kernels.upload_plan(plan, gpu), ctx,
                                          types.SimpleNamespace(block_table=bt.to(gpu)), kv, HEADS, D**-0.5, window, rule)
        got = got.double().cpu().view(-1, HEADS, D)
        # every weight is rounded to 8 bits (2^-9 of it), and the result; as much again for the exponentials and the order of the sums
        assert bool(((got - want).abs() <= 2.0**-7 * size).all()), float(((got - want).abs() / size.clamp(min=1e-30)).max())
