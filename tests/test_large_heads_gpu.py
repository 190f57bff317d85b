"""Attention with heads of more than 128 dimensions: the kernel for long segments (values whose
first quarter of dimensions is zeros have a build of their own at 256), and the rule that says when
a step's long segments go to it."""

import types

import numpy as np
import pytest
import torch

from halite_amd.kernels import attention as attn_kernels
from test_kernels_gpu import paged_cache, rnd, to_tiled

import plain_llama as P

FROM = 64


def case(gpu, H, K, D, page, segs, window, tiled, value_from, seed, poison):
    """Segments (tokens before, new tokens) against the plain attention; ``poison``: the values' first
    dimensions are NaN in the pages, so that a kernel that reads them shows."""
    dt = torch.bfloat16
    qs, ks, vs, rows, want, base = [], [], [], [], [], 0
    for i, (before, new) in enumerate(segs):
        n = before + new
        q, k, v = (rnd(n, h, D, seed=seed + 3 * i + j).to(dt).float() for j, h in enumerate((H, K, K)))
        if n > 40:  # one far key stands out: a kernel that drops or misplaces it shows
            k[3], q[-1], v[3] = 0, 0, 5.0
            k[3, :, 0], q[-1, :, 0] = 6.0, 2.0 * D**0.5
        v[..., :value_from] = 0
        want.append(P.causal_attention(q, k, v, window=window or None)[before:].reshape(new, H * D))
        qs.append(q[before:].reshape(new, H * D))
        if poison:
            v[..., :value_from] = float("nan")
        kp, vp, row = paged_cache(k, v, page, seed + i, dtype=dt)
        ks.append(kp), vs.append(vp), rows.append(row + base)
        base += kp.shape[0]
    bt = torch.full((len(segs), max(len(r) for r in rows)), -1, dtype=torch.int32)
    for i, r in enumerate(rows):
        bt[i, : len(r)] = r
    k_pages, v_pages = torch.cat(ks), torch.cat(vs)
    if tiled:
        k_pages, v_pages = to_tiled(k_pages, v_pages)
    q_len = np.array([n for _, n in segs], dtype=np.int32)
    kv_len = np.array([b + n for b, n in segs], dtype=np.int32)
    rows_big = attn_kernels.rows_per_big_item(D, value_from)
    out = []
    for r in {rows_big, attn_kernels.ROWS_PER_ITEM}:  # the kernel for long segments, and one-tile items alone
        plan = attn_kernels.plan_items(q_len, kv_len, H // K, K, window, r)
        dev = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(gpu)  # noqa: E731
        starts = np.concatenate(([0], np.cumsum(q_len)[:-1])).astype(np.int32)
        ctx = types.SimpleNamespace(n_tokens=int(q_len.sum()), seg_q_start=dev(starts), seg_q_len=dev(q_len), seg_kv_len=dev(kv_len))
        kv = types.SimpleNamespace(k=k_pages.to(gpu), v=v_pages.to(gpu), tiled=tiled, value_from=value_from)
        got = attn_kernels.attention_mfma(torch.cat(qs).to(dt).to(gpu), H * D, attn_kernels.upload_plan(plan, gpu), ctx,
                                          types.SimpleNamespace(block_table=bt.to(gpu)), kv, H, D**-0.5, window)
        # probabilities and results are rounded to 8 bits: 2^-8 of the largest value (5) each
        assert float((got.float().cpu() - torch.cat(want)).abs().max()) < 2 * 5 * 2.0**-8
        zeros = got.view(-1, H, D)[..., :value_from]
        assert bool((zeros == 0).all())
        out.append(plan.n_big)
    return out


SEGS = [[(0, 1)], [(0, 70)], [(63, 1), (0, 33), (64, 64), (129, 2), (200, 1)], [(700, 1), (5, 300)], [(2000, 1), (900, 1), (1199, 2)]]


@pytest.mark.gpu
@pytest.mark.parametrize("segs", SEGS)
@pytest.mark.parametrize("H, K", [(32, 1), (6, 3), (5, 1)])
def test_values_that_begin_behind_zeros(H, K, segs):
    gpu = torch.device("cuda:0")
    for page, window, tiled in ((16, 0, False), (64, 0, True), (24, 0, False), (64, 300, True), (64, 37, False)):
        n_big = case(gpu, H, K, 256, page, segs, window, tiled, FROM, 50, poison=True)
        assert len(n_big) == 2 and (max(n_big) > 0) == any(new > 1 and new * (H // K) > 16 for _, new in segs)


@pytest.mark.gpu
@pytest.mark.parametrize("D", [160, 256])
def test_values_from_without_a_build_of_its_own(D):
    """Fewer zeros than the build skips, or another head size: all dimensions are read."""
    gpu = torch.device("cuda:0")
    n_big = case(gpu, 8, 2, D, 64, [(300, 90), (0, 40), (9, 1)], 0, True, 32, 60, poison=False)
    assert (max(n_big) > 0) == (D <= 224)


def test_when_long_items_pay():
    pay = attn_kernels.long_items_pay
    assert pay([2], [2], 1, 1, 0, 128)  # up to 128 dimensions always
    # a latent's one key/value head: by (row, key) pairs, tokens that see few keys of a window counted so
    assert pay([1024], [1024], 16, 1, 0, 256, 64) and not pay([512], [512], 16, 1, 0, 256, 64)
    assert pay([64], [4160], 32, 1, 0, 256, 64) and not pay([64], [4160], 32, 1, 100, 256, 64)
    assert not pay([1] * 64, [8192] * 64, 32, 1, 0, 256, 64)  # decode tokens are never long segments
    # values in all dimensions: a workgroup a compute unit besides
    assert pay([2048], [2048], 4, 4, 0, 160) and not pay([2048], [2048], 1, 8, 0, 160)
