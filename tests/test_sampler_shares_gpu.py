"""Rows whose lists and kept masses are put together by many threads: the same draw every time, alone and beside others, and against 64 bits
where a list is longer than what the last kernel holds of it, or empty."""

import numpy as np
import pytest
import torch

from halite_amd.sampling import Sampler, SamplingParams

pytestmark = pytest.mark.gpu

WAYS = [dict(top_p=0.9), dict(top_k=50), dict(min_p=0.05), dict(top_k=50, top_p=0.9, min_p=0.02), dict(top_p=1e-9), dict(top_k=4096, top_p=0.999)]


@pytest.mark.parametrize("vocab", [33, 4095, 4096, 9001, 50257])
@pytest.mark.parametrize("spread", [0.02, 2.0])
def test_the_same_draw_every_time(vocab, spread):
    x = (torch.randn((24, vocab), generator=torch.Generator().manual_seed(vocab)) * spread).cuda()
    params = [SamplingParams(temperature=0.8, **WAYS[r % len(WAYS)]) for r in range(24)]
    seeds, draws, sampler = list(range(24)), [r + 3 for r in range(24)], Sampler("cuda")
    tokens, logprobs = sampler.forward(x, params, seeds, draws)
    for _ in range(5):
        again, again_lp = sampler.forward(x, params, seeds, draws)
        assert torch.equal(tokens, again) and torch.equal(logprobs, again_lp)
    for r in (0, 3, 17):
        alone, alone_lp = sampler.forward(x[r : r + 1], params[r : r + 1], seeds[r : r + 1], draws[r : r + 1])
        assert int(alone) == int(tokens[r]) and float(alone_lp) == float(logprobs[r])


@pytest.mark.parametrize("vocab", [4097, 20000])
@pytest.mark.parametrize("spread", [0.0, 0.02, 1.0])
def test_draws_come_from_what_is_kept(vocab, spread):
    """Every drawn token is among the most likely ones that top-p of 64-bit masses keeps (one more, where the sum is within rounding of
    its target), and its log-probability is right."""
    n = 64
    x = torch.randn((n, vocab), generator=torch.Generator().manual_seed(7)) * spread
    top_p = [0.3, 0.9, 0.999][:3]
    params = [SamplingParams(temperature=1.0, top_p=top_p[r % 3]) for r in range(n)]
    tokens, logprobs = (t.cpu().numpy() for t in Sampler("cuda").forward(x.cuda(), params, list(range(n)), [0] * n))
    p = torch.softmax(x.double(), dim=1).numpy()
    for r in range(n):
        order = np.sort(p[r])[::-1]
        kept = int(np.searchsorted(np.cumsum(order), params[r].top_p)) + 1
        assert p[r, tokens[r]] >= order[min(kept, vocab - 1)] * (1 - 1e-6)  # (ties at the threshold are all kept)
        assert abs(logprobs[r] - np.log(p[r, tokens[r]])) < 1e-5
