"""What the model's last product is told of the final norm: nothing, unless the norm, the block and its feed-forward all
say that they know of sums that the norm adds up; and no block or norm with the plain interface is asked for more."""

from types import SimpleNamespace

import pytest
import torch

from halite_amd.kernels import ops
from halite_amd.parts.base import Arrangement, FeedForward, Norm
from halite_amd.parts.block import PreNormBlock
from halite_amd.parts.decoder import Decoder


class PlainNorm(Norm):
    def __init__(self):
        self.got = []

    def forward(self, h, delta=None, rows=None):
        self.got.append((delta, rows))
        return h if rows is None else h[rows.long()]

    def foldable(self, h):
        return None


class FoldedNorm(PlainNorm):
    def foldable(self, h):
        return ops.NextNorm(h, torch.ones(h.shape[1]), 1e-5)


class SummingNorm(PlainNorm):
    def summable(self, h):
        return ops.NextNorm(h, torch.ones(h.shape[1]), 1e-5, sums=True, gathers=True)


class Part(FeedForward):
    def __init__(self, folds=False, leaves=False):
        self.folds_next_norm, self.leaves_sums, self.told = folds, leaves, []

    def forward(self, x, ctx, run=None, then=None):
        self.told.append(then)
        return x


class OwnBlock(Arrangement):
    takes_next_norm = True

    def __init__(self):
        self.told = []

    def forward(self, h, pending, ctx, run, next_norm=None):
        self.told.append(next_norm)
        return pending


def model(blocks, final_norm):
    d = Decoder.__new__(Decoder)
    h = torch.zeros((3, 4))
    d.embedding = SimpleNamespace(reads_step=False, forward=lambda tokens: h)
    d.layers = dict(enumerate(blocks))
    d.spec = SimpleNamespace(order=[SimpleNamespace(layer=i, junction=None) for i in range(len(blocks))], hidden_size=4, vocab_size=4)
    d.runs = [SimpleNamespace(index=i) for i in range(len(blocks))]
    d.junctions, d.stream_copies, d.device, d.final_norm = {}, None, torch.device("cpu"), final_norm
    d.head = SimpleNamespace(forward=lambda x: x)
    return d


def step(blocks, final_norm):
    ctx = SimpleNamespace(tokens=torch.zeros(3, dtype=torch.int32), n_logit_rows=1, logit_rows=torch.tensor([2], dtype=torch.int32))
    return model(blocks, final_norm).forward(ctx)


def block(ff):
    return PreNormBlock(dict(mixer_norm=PlainNorm(), mixer=Part(), ff_norm=PlainNorm(), ff=ff))


@pytest.mark.parametrize("norm", [PlainNorm, FoldedNorm, SummingNorm])
@pytest.mark.parametrize("folds, leaves", [(False, False), (True, False), (True, True)])
def test_who_is_told(norm, folds, leaves):
    parts = [Part(folds, leaves), Part(folds, leaves)]
    final = norm()
    step([block(ff) for ff in parts], final)
    told = parts[1].told[0]
    if norm is SummingNorm and leaves:
        assert told.sums and told.gathers
    else:
        assert told is None
    assert parts[0].told == [None] and len(final.got) == 1


@pytest.mark.parametrize("norm", [PlainNorm, FoldedNorm, SummingNorm])
def test_an_arrangement_with_the_plain_interface(norm):
    own = OwnBlock()
    step([own], norm())
    assert own.told == [None]


def test_results_that_are_wanted_in_float32_come_whole():
    """(the choice itself, without a GPU: only 16-bit results may come in parts, since the reader rounds their sum)"""
    seen = []

    def parts(x, w, n, gated=False, may_part=False):
        seen.append(may_part)
        raise StopIteration

    x, w = torch.zeros((17, 64), dtype=torch.bfloat16), torch.zeros((128, 64), dtype=torch.bfloat16)
    norm = ops.NextNorm(torch.zeros((17, 128)), torch.ones(128), 1e-5, sums=True, gathers=True)
    kept, ops.stream_parts = ops.stream_parts, parts
    try:
        for how in (dict(sums=True), dict(next_norm=norm), dict(sums=True, out_dtype=torch.float32), dict(next_norm=norm, out_dtype=torch.float32)):
            with pytest.raises(StopIteration):
                ops.linear(x, w, **how)
    finally:
        ops.stream_parts = kept
    assert seen == [True, True, False, False]
