"""A step's sampling parameters in one buffer, against their packing by numpy (no GPU is needed)."""

import random

import numpy as np
import pytest
import torch

from halite_amd.kernels import ops
from halite_amd.sampling import SamplingParams
from halite_amd.sampling.sampler import Sampler, _integers, array


def by_numpy(params, seeds, draws, vocab):
    n = len(params)
    words = np.empty(7 * n, np.int32)
    words[: 2 * n].view(np.int64)[:] = seeds
    f, i = words[2 * n : 5 * n].view(np.float32).reshape(3, n), words[5 * n :].reshape(2, n)
    temperature, top_k = np.array([p.temperature for p in params], np.float64), np.array([p.top_k for p in params])
    top_p, min_p = np.array([p.top_p for p in params], np.float64), np.array([p.min_p for p in params], np.float64)
    greedy = (temperature == 0) | (top_k == 1)
    f[0], f[1], f[2] = np.where(greedy, 0.0, temperature), top_p, min_p
    i[0], i[1] = np.where(greedy, 1, np.minimum(top_k, 2**31 - 1)), draws
    by_k, by_p, by_min = (top_k > 0) & (top_k < vocab), top_p < 1.0, min_p > 0.0
    unfiltered, late = not np.any(~greedy & (by_k | by_p | by_min)), bool(np.any(~greedy & by_k & by_p & by_min))
    return words, (1 if greedy.all() else 0) | (2 if unfiltered else 0) | (4 if late else 0)


@pytest.mark.parametrize("n,seed", [(1, 0), (2, 1), (7, 2), (64, 3), (64, 4), (1000, 5)])
@pytest.mark.parametrize("kind", ["greedy", "whole", "top_p", "mixed"])
def test_as_numpy_packs_them(n, seed, kind):
    rng = random.Random(seed)
    pick = dict(greedy=dict(temperature=[0, 0.0], top_k=[1, -1, 40]), whole=dict(temperature=[0.0, 0.7, 1], top_k=[-1, 50257, 2**40, 10**30 if seed == 1 else 1]),
                top_p=dict(temperature=[0.8], top_p=[0.9]),
                mixed=dict(temperature=[0.0, 1e-9, 0.3, 2], top_k=[-1, 1, 2, 50, 50256], top_p=[1, 1e-12, 1 - 2.0**-40, 0.5], min_p=[0, 1e-30, 0.1, 1]))[kind]
    params = [SamplingParams(**{k: rng.choice(v) for k, v in pick.items()}) for _ in range(n)]
    seeds, draws = [rng.choice([0, 1, 2**63 - 1, -(2**63), rng.getrandbits(62)]) for _ in range(n)], [rng.choice([0, 5, 2**31 - 1]) for _ in range(n)]
    want, flags = by_numpy(params, seeds, draws, 50257)
    host = torch.empty(7 * n + 3, dtype=torch.int32)
    got = ops.pack_sample_rows(host, *(array("d", [getattr(p, k) for p in params]) for k in ("temperature", "top_p", "min_p")),
                               _integers([p.top_k for p in params], 2**31 - 1), _integers(seeds), _integers(draws), 50257)
    assert got == flags and np.array_equal(host.numpy()[: 7 * n], want)


def test_other_numbers_than_integers():
    assert _integers([np.int32(3), 2.0, 4], 10).tolist() == [3, 2, 4] and _integers(np.array([1, 2])).tolist() == [1, 2]
    assert _integers([10**30, 5], 7).tolist() == [7, 5]
    with pytest.raises(OverflowError):
        _integers([10**30])


@pytest.mark.parametrize("bad", [2**63, 2**63 + 5, -(2**63) - 1, 2**64])
def test_seeds_out_of_range_are_refused(bad):
    """Rounded or wrapped, two of them could become one."""
    for values in ([bad], [bad, 1], [1, bad], [bad, -1]):
        with pytest.raises(OverflowError):
            _integers(values)


@pytest.mark.parametrize("bad", [2**31, -(2**31) - 1, 2**32 + 3, 2**63])
def test_draws_out_of_range_are_refused(bad):
    with pytest.raises(OverflowError):
        ops.pack_sample_rows(torch.empty(14, dtype=torch.int32), *[array("d", [0.5, 0.5])] * 3, *[array("q", [1, 1])] * 2, _integers([0, bad]), 50)


def test_sampler_refuses_them():
    if not torch.cuda.is_available():
        sampler = Sampler("cpu")
        sampler._stage = lambda words: torch.empty(words, dtype=torch.int32)  # (no pinned memory without a GPU)
    else:
        sampler = Sampler("cuda:0")
    logits = torch.zeros((2, 5), device=sampler.device)
    for seeds, draws in (([2**63 + 5, 1], [0, 0]), ([1, 2], [0, 2**31])):
        with pytest.raises(OverflowError):
            sampler.forward(logits, [SamplingParams(), SamplingParams()], seeds, draws)


def test_arrays_of_other_lengths_and_types_are_refused():
    """Six entries each are read from them."""
    good = [array("d", [0.5] * 6)] * 3 + [array("q", [1] * 6)] * 3
    host = torch.empty(42, dtype=torch.int32)
    ops.pack_sample_rows(host, *good, 50)
    for i in range(6):
        for bad in (good[i][:5], good[i][:0], array("f" if i < 3 else "i", [1] * 6), array("q" if i < 3 else "d", [1] * 6), [1] * 6):
            with pytest.raises(ops.KernelError):
                ops.pack_sample_rows(host, *good[:i], bad, *good[i + 1 :], 50)
    with pytest.raises(ops.KernelError):
        ops.pack_sample_rows(host[:41], *good, 50)
