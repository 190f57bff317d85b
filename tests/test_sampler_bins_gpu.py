"""Filters found by bins of the distance from the maximum and a list of one bin's keys, against the one-block kernel
(which selects by the keys' bits): lists of one key, of more than LDS holds and of all keys, thresholds in the last bin,
equal logits, masked and infinite ones, temperatures at the type's ends, rows of every kind side by side."""

import random

import pytest
import torch

from halite_amd.kernels import ops

pytestmark = pytest.mark.gpu


def both(x, temperature, top_k, top_p, min_p, seed):
    n = x.shape[0]
    f = lambda v: torch.tensor(v, dtype=torch.float32, device=x.device)  # noqa: E731
    args = (f(temperature), torch.tensor(top_k, dtype=torch.int32, device=x.device), f(top_p), f(min_p),
            torch.arange(n, dtype=torch.int64, device=x.device) * 7919 + seed, torch.arange(n, dtype=torch.int32, device=x.device))
    return [[t.cpu() for t in ops.sample(x, *args, spread=spread)] for spread in (False, True)]


def agree(ways, rows, allowed=0):
    (tok, lp), (tok2, lp2) = ways
    same = tok == tok2
    assert int((~same).sum()) <= allowed, (tok[~same].tolist(), tok2[~same].tolist())
    assert torch.equal(lp.isnan(), lp2.isnan())
    # (sums of up to 2e5 float32 exponentials in two orders, and their logarithm)
    assert torch.allclose(lp[same & ~lp.isnan()], lp2[same & ~lp.isnan()], rtol=1e-5, atol=1e-5)
    assert same.numel() == rows


@pytest.mark.parametrize("vocab", [1, 2, 255, 4097, 32000, 131073])
@pytest.mark.parametrize("spread", [0.01, 1.0, 30.0])
def test_drawn_rows(vocab, spread):
    """Where the draw falls within rounding of a token's edge the two may differ: a chance of some 1e-7 a kept token and
    row, so one row in a hundred at most."""
    rng, n = random.Random(vocab), 100
    gen = torch.Generator().manual_seed(vocab)
    x = (torch.randn((n, vocab), generator=gen) * spread)
    x[::7] = x[::7].to(torch.bfloat16).float()  # many equal logits
    x[1::7, ::3] = -float("inf")
    ways = both(x.cuda(), [rng.choice([0.0, 0.1, 0.7, 1.0, 2.5]) for _ in range(n)],
                [rng.choice([-1, -1, 1, 2, 40, max(1, vocab - 1), vocab, vocab + 5]) for _ in range(n)],
                [rng.choice([0.01, 0.3, 0.9, 0.999, 1.0]) for _ in range(n)], [rng.choice([0.0, 0.0, 0.05, 1.0]) for _ in range(n)], 3)
    agree(ways, n, allowed=1)


@pytest.mark.parametrize("rows_at_once", [1, 3, 7, 20, 21])
def test_rows_in_turns(monkeypatch, rows_at_once):
    """More rows than there is room for lists: the same tokens, turn by turn over one room."""
    n, vocab, rng = 20, 5000, random.Random(5)
    x = torch.randn((n, vocab), generator=torch.Generator().manual_seed(2)).cuda()
    params = ([rng.choice([0.0, 0.7, 1.0]) for _ in range(n)], [rng.choice([-1, 1, 40, 4999]) for _ in range(n)],
              [rng.choice([0.3, 0.9, 1.0]) for _ in range(n)], [rng.choice([0.0, 0.05]) for _ in range(n)], 11)
    (_, _), (tok, lp) = both(x, *params)
    monkeypatch.setattr(ops, "SAMPLE_LIST_WORDS", rows_at_once * vocab + 1)
    (_, _), (tok2, lp2) = both(x, *params)
    assert torch.equal(tok, tok2) and torch.equal(lp, lp2)


@pytest.mark.parametrize("kind", ["greedy", "whole", "filtered", "late at the end"])
@pytest.mark.parametrize("n, rows_at_once", [(1, 1), (20, 1), (20, 7), (21, 7), (22, 7), (23, 64)])
def test_as_the_engine_samples(monkeypatch, kind, n, rows_at_once):
    """The sampler with its requests' own parameters, rows in turns over one room, a cut last turn, the only row with all
    three filters in it: the tokens of the one-block kernel."""
    from halite_amd.sampling import SamplingParams
    from halite_amd.sampling.sampler import Sampler

    vocab, rng = 5000, random.Random(n + rows_at_once)
    x = (torch.randn((n, vocab), generator=torch.Generator().manual_seed(n)) * 2).cuda()
    pick = {"greedy": dict(temperature=[0.0, 0.7], top_k=[1]), "whole": dict(temperature=[0.0, 0.3, 1.0, 2.0]),
            "filtered": dict(temperature=[0.0, 0.7, 1.0], top_k=[-1, 1, 40, 6000], top_p=[0.3, 0.9, 1.0]),
            "late at the end": dict(temperature=[0.7, 1.0], top_k=[-1, 40], min_p=[0.0, 0.05])}[kind]
    params = [SamplingParams(**{k: rng.choice(v) for k, v in pick.items()}) for _ in range(n)]
    if kind == "late at the end":
        params[-1] = SamplingParams(temperature=0.9, top_k=30, top_p=0.8, min_p=0.01)
    seeds, draws = [rng.getrandbits(62) for _ in range(n)], [rng.randrange(1000) for _ in range(n)]
    f = lambda v, dt=torch.float32: torch.tensor(v, dtype=dt, device="cuda")  # noqa: E731
    want = ops.sample(x, f([p.temperature for p in params]), f([p.top_k for p in params], torch.int32), f([p.top_p for p in params]),
                      f([p.min_p for p in params]), f(seeds, torch.int64), f(draws, torch.int32))
    monkeypatch.setattr(ops, "SAMPLE_LIST_WORDS", rows_at_once * vocab + 1)
    sampler = Sampler("cuda:0")
    for _ in range(2):  # (the second time over a staging buffer of its own)
        agree([[t.cpu() for t in want], [t.cpu() for t in sampler.forward(x, params, seeds, draws)]], n)
    assert sampler.forward(x[:0], [], [], [])[0].numel() == 0


def test_no_rows():
    x = torch.zeros((0, 50), device="cuda")
    for flags in range(8):
        tok, lp = ops.sample_packed(x, torch.zeros(0, dtype=torch.int32, device="cuda"), flags)
        assert tok.numel() == lp.numel() == 0


def test_room_for_many_rows():
    """What a step holds beside its logits does not grow with them: 256 MiB of lists, and 5 KiB a row of the rows in turn."""
    n, vocab = 1100, 100000
    x = torch.zeros((n, vocab), device="cuda")
    full = lambda v, dt=torch.float32: torch.full((n,), v, dtype=dt, device="cuda")  # noqa: E731
    args = (full(1.0), full(-1, torch.int32), full(0.9), full(0.0), full(1, torch.int64), full(1, torch.int32))
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    torch.cuda.reset_peak_memory_stats()
    before = torch.cuda.memory_allocated()
    ops.sample(x, *args, spread=True)
    assert torch.cuda.max_memory_allocated() - before < 272 * 2**20


def test_rows_at_the_ends():
    n, vocab = 12, 6000
    x = torch.randn((n, vocab), generator=torch.Generator().manual_seed(1))
    x[0] = 0.0                                     # all equal: the list is the row
    x[1], x[1, 17], x[1, 4000] = -float("inf"), 1.0, 1.0
    x[2] = -float("inf")                           # nothing
    x[3, 40], x[3, 700] = float("inf"), float("inf")
    x[4, ::2] = float("nan")
    x[5] = torch.linspace(0, -200, vocab)          # most keys in the last bin
    x[6] = torch.linspace(0, -200, vocab)
    x[7] = x[7] * 1e-38                            # quotients that are no normal numbers
    x[8] = x[8] * 1e30
    x[9, 100:] = x[9, 0]                           # one key and many of another
    temperature = [1.0] * n
    temperature[7], temperature[8] = 100.0, 1e-9   # ... and such that overflow
    top_k = [3000, -1, 5, 5, -1, 5500, -1, 50, 50, 200, 1, -1]
    top_p = [1.0, 0.4, 0.9, 0.9, 0.9, 1.0, 0.5, 0.9, 0.9, 0.9, 0.5, 0.0]
    for seed in range(8):
        agree(both(x.cuda(), temperature, top_k, top_p, [0.0] * n, seed), n)
        agree(both(x.cuda(), temperature, top_k, top_p, [0.001] * n, seed), n)
