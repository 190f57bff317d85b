"""Float32 attention of prompts: waves that share the rows and split the keys where a step has up to 256 workgroups, and
waves that have their rows to themselves where it has more."""

import pytest
import torch
from test_kernels_gpu import attention_case

from halite_amd.kernels import ops

pytestmark = pytest.mark.gpu


# 32 tokens a workgroup times 8 heads of keys: 256 workgroups and 264 (and 304 of 128 tokens); several requests in one workgroup; portions
@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("H, K, D, segs", [(32, 8, 128, [(0, 1024)]), (32, 8, 128, [(0, 1025)]), (32, 8, 96, [(70, 1060)]), (16, 16, 64, 9 * [(0, 260)]),
                                           (32, 8, 72, [(0, 33), (31, 34), (63, 9), (64, 130), (500, 40)]), (12, 4, 128, [(0, 300), (129, 31)])])
def test_split_and_whole(dtype, H, K, D, segs):
    for page, window in ((16, 0), (64, 37)):
        attention_case(torch.device("cuda:0"), dtype, H, K, D, page, segs, window, seed=31, use="simple")


# a request alone (up to 256 workgroups) and beside others that make them more: the same numbers, bit for bit; several
# requests share a workgroup, and the request's rows and blocks lie elsewhere in it
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("window, keep", [(0, 0), (37, 0), (150, 5)])
@pytest.mark.parametrize("H, K, D, before, new", [(32, 8, 128, 0, 300), (32, 8, 72, 700, 75), (16, 16, 64, 70, 260), (12, 4, 96, 33, 129), (8, 1, 24, 5, 1000)])
def test_what_else_is_in_the_step(H, K, D, before, new, window, keep, dtype):
    page, gpu, gen = 16, torch.device("cuda:0"), torch.Generator().manual_seed(D)
    rand = lambda *shape: torch.randn(*shape, generator=gen).to(dtype)  # noqa: E731
    others = 4 if K > 4 else 9
    segs = [(0, 45), (before, new)] + [(3, 1021)] * others
    pages = [-(-(b + n) // page) for b, n in segs]
    firsts = [sum(pages[:i]) for i in range(len(segs))]
    tables = torch.full((len(segs), max(pages)), -1, dtype=torch.int32)
    for i, n in enumerate(pages):
        tables[i, :n] = torch.arange(firsts[i], firsts[i] + n)
    k_pages, v_pages = rand(sum(pages), K, page, D).to(gpu), rand(sum(pages), K, D, page).to(gpu)
    q = [rand(n, H * D) for _, n in segs]

    def rows(which):
        i32 = lambda t: t.to(torch.int32).to(gpu)  # noqa: E731
        out = ops.attention_simple(
            torch.cat([q[i] for i in which]).to(gpu), H * D, i32(torch.cat([torch.arange(segs[i][0], sum(segs[i])) for i in which])),
            i32(torch.cat([torch.full((segs[i][1],), j) for j, i in enumerate(which)])), tables[which].to(gpu), k_pages, v_pages, H, D**-0.5, window,
            max_kv_len=max(sum(segs[i]) for i in which), min_q_len=min(segs[i][1] for i in which), rule=ops.ScoreRule(keep=keep))
        at = sum(segs[i][1] for i in which[: which.index(1)])
        return out[at : at + new]

    groups = lambda which: -(-sum(segs[i][1] for i in which) // max(1, 128 // (H // K))) * K  # noqa: E731
    everything = list(range(len(segs)))
    assert groups([1]) <= 256 < groups(everything)
    alone = rows([1])
    assert torch.equal(alone, rows([0, 1])) and torch.equal(alone, rows(everything))
