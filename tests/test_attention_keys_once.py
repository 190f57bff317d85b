"""Whether the attention kernel for one-tile items is told that a step reads its keys once, without a GPU."""

from types import SimpleNamespace

import numpy as np
import pytest
import torch

from halite_amd.kernels import attention as attn_kernels


# (segments' new tokens, heads of a key head, rows of a long item) -> whether every one-tile segment is one tile
@pytest.mark.parametrize("q_len, group, rows_big, once", [([1, 1], 4, 64, True), ([1], 16, 16, True), ([1, 1], 32, 64, False), ([4, 1], 4, 64, True), ([5, 1], 4, 16, False),
                                                          ([1, 500], 16, 16, False), ([500], 16, 64, True), ([1, 2000, 1], 4, 64, True), ([17], 1, 16, False), ([16, 16], 1, 16, True), ([], 4, 64, True)])
def test_keys_that_a_step_reads_once(monkeypatch, q_len, group, rows_big, once):
    """The kernel is told what the plan says, whatever the heads: a segment of several tiles has its keys read by each."""
    plan = attn_kernels.plan_items(np.array(q_len, dtype=np.int32), np.array(q_len, dtype=np.int32) + 900, group, 2, 0, rows_big)
    assert plan.keys_once == once
    told = []
    monkeypatch.setattr(attn_kernels.library, "attention_library", lambda d: SimpleNamespace(hal_attention_mfma_ruled=lambda *a: told.append(a[-3]) or 0))
    monkeypatch.setattr(attn_kernels.ops, "_stream", lambda: None)
    monkeypatch.setattr(attn_kernels, "_counters", lambda device: None)
    heads, n = 2 * group, sum(q_len)
    ctx = SimpleNamespace(n_tokens=n, seg_q_start=None, seg_q_len=None, seg_kv_len=None)
    kv = SimpleNamespace(k=torch.zeros(1, 2, 64, 256), v=torch.zeros(1, 2, 64, 256), tiled=True)
    attn_kernels.attention_mfma(torch.zeros(n, heads * 256), heads * 256, (plan, None, None, None, None), ctx, SimpleNamespace(block_table=torch.zeros(1, 1)), kv, heads, 1.0, 0)
    assert told == [1 if once else 0]
