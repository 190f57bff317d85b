"""Which products the wide tiles are asked for, without a GPU: what their entry point refuses goes where it went before them."""

from types import SimpleNamespace

import pytest
import torch

from halite_amd.kernels import ops


def rows(m, k, apart, place=0, step=1, dtype=torch.bfloat16):
    return SimpleNamespace(shape=(m, k), dtype=dtype, is_cuda=True, stride=lambda: (apart, step), data_ptr=lambda: 1 << 20 | place)


def takes(m, n, k, x=None, w=None, **how):
    return ops.wide_pays(x or rows(m, k, k), w or rows(n, k, k), n, **how)


@pytest.mark.parametrize("m, n, k", [(2048, 4096, 4096), (2048, 4100, 4096), (1000, 6144, 4096), (500, 6144, 1536)])
def test_places_and_distances(m, n, k):
    assert takes(m, n, k) and takes(m, n, k, x=rows(m, k, k + 8)) and takes(m, n, k, w=rows(n, k, 2**21 - 8))
    for of_x in (True, False):
        a, which = (m, "x") if of_x else (n, "w")
        for other in (rows(a, k, k, place=8), rows(a, k, k + 4), rows(a, k, 2**21), rows(a, k, 2**31), rows(a, k, 0), rows(a, k, 1, step=a), rows(a, k, k - 8),
                      rows(a, k, k, dtype=torch.float32)):
            assert not takes(m, n, k, **{which: other})


def test_sizes():
    assert not takes(64, 14336, 4096, gated=True) and takes(500, 14336, 4096, gated=True)
    assert not takes(2048, 4098, 4096) and not takes(2048, 4096, 4096 + 64) and not takes(2048, 4096, 4000)
    assert takes(2048, 4096, 128) == takes(2048, 4096, 128, x=rows(2048, 128, 136)) and not takes(2048, 4096, 64)


def test_what_the_answer_hangs_on_is_kept_for_it():
    """Answers are kept for sizes and distances, so that a matrix of the same size with rows elsewhere has its own."""
    for x, want in ((rows(2048, 4096, 4096), True), (rows(2048, 4096, 4100), False), (rows(2048, 4096, 4104), True), (rows(2048, 4096, 4096, step=2), False)):
        assert takes(2048, 4096, 4096, x=x) == want


def test_tensors_on_the_host_ask_no_library(monkeypatch):
    def asked(*sizes):
        raise AssertionError("asked for the library")

    monkeypatch.setattr(ops, "_wide_pays", asked)
    x, w = torch.randn(2048, 128).bfloat16(), torch.randn(4096, 128).bfloat16()
    assert not ops.wide_pays(x, w, 4096) and torch.equal(ops.linear(x, w), x @ w.t())
