"""The sampler's passes over a row spread over many blocks: vocabularies at which a block's share begins
another load a thread, the last of a batch of them, a second batch."""

import pytest
import torch

import plain_llama as P
from halite_amd.kernels import ops
from test_kernels_gpu import _sample, rnd

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("vocab", [1, 33, 8192, 8193, 122880, 122881, 131072, 131073, 262147])
def test_shares(vocab):
    gpu, n = torch.device("cuda:0"), 12
    base = rnd(1, vocab, seed=vocab, scale=3.0)[0]
    base[-1] = base.max() + 2.0  # the very last logit counts
    logits = base[None].repeat(n, 1)
    full = lambda v, dt: torch.full((n,), v, dtype=dt, device=gpu)  # noqa: E731
    for kw in ({"top_p": 0.9, "temperature": 0.8}, {"top_k": 40, "top_p": 0.9, "min_p": 0.01}, {}):
        params = {"temperature": 1.0, "seed": 5, **kw}
        if kw:
            tok, lp = _sample(gpu, logits, seed=5, spread=True, **kw)
        else:
            tok, lp = ops.sample(logits.to(gpu), full(1.0, torch.float32), full(-1, torch.int32), full(1.0, torch.float32), full(0.0, torch.float32),
                                 full(5, torch.int64), torch.arange(n, dtype=torch.int32, device=gpu), unfiltered=True)
        agree = 0
        for i in range(n):
            t, logprob, margin = P.sample_token(base, params, i)
            if margin > 2e-5:  # (a draw this close to a token's edge may fall to its neighbour)
                assert int(tok[i]) == t and abs(float(lp[i]) - logprob) < 2e-4, (kw, i)
                agree += 1
        assert agree >= n // 2
    greedy, _ = ops.sample(logits.to(gpu), full(0.0, torch.float32), full(-1, torch.int32), full(1.0, torch.float32), full(0.0, torch.float32),
                           full(5, torch.int64), full(0, torch.int32), all_greedy=True)
    assert greedy.tolist() == [vocab - 1] * n
