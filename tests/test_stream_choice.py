"""Which products the streaming kernel is asked for, without a GPU: rows so far apart that its 32-bit offsets do not reach
them go where they went before it."""

from types import SimpleNamespace

import pytest
import torch

from halite_amd.kernels import ops


def rows(m, k, apart, place=0):
    return SimpleNamespace(shape=(m, k), dtype=torch.bfloat16, is_cuda=True, stride=lambda d: (apart, 1)[d], data_ptr=lambda: 1 << 20 | place)


@pytest.mark.parametrize("m, apart, takes", [(64, 4096, True), (64, 2**24 - 8, True), (64, 2**24, False), (17, 2**30 // 17 // 8 * 8, True),
                                             (17, 2**30 // 17 // 8 * 8 + 8, False), (16, 4096, False), (65, 4096, False)])
def test_rows_far_apart(monkeypatch, m, apart, takes):
    monkeypatch.setattr(ops, "_stream_parts", lambda *sizes: 4)
    assert bool(ops.stream_parts(rows(m, 4096, apart), rows(4096, 4096, 4096), 4096, may_part=True)) == takes


def test_places(monkeypatch):
    monkeypatch.setattr(ops, "_stream_parts", lambda *sizes: 4)
    w = rows(4096, 4096, 4096)
    assert ops.stream_parts(rows(33, 4096, 4096), w, 4096) == 4
    assert not ops.stream_parts(rows(33, 4096, 4096, place=8), w, 4096) and not ops.stream_parts(rows(33, 4096, 4100), w, 4096)
    assert not ops.stream_parts(rows(33, 4096, 4096), rows(4096, 4096, 4096, place=2), 4096)
    assert not ops.stream_parts(rows(33, 4096, 4096), rows(4096, 4096, 2**18), 4096)  # (2 GiB of weights)
