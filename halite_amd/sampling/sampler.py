"""The sampler on top of the sampling kernel
(src/halite/transformers/infer/engine/sampler.py:12-60)."""

from __future__ import annotations

import zlib
from array import array

import numpy as np
import torch

from ..kernels import ops
from .params import SamplingParams

_MASK63 = (1 << 63) - 1


def request_seed(params: SamplingParams, request_id, engine_seed: int = 0) -> int:
    """The seed of a request's random stream: its own if given, else derived from
    the engine's seed and the request's id, so that it does not depend on what else
    runs."""
    if params.seed is not None:
        return int(params.seed) & _MASK63
    return (zlib.crc32(repr(request_id).encode()) * 2654435761 + engine_seed * 40503) & _MASK63


def _integers(values, most: int | None = None) -> array:
    """Whole numbers as 64-bit integers; one that is out of their range raises ``OverflowError`` (``most``: larger ones
    count as that)."""
    try:
        return array("q", values)
    except (TypeError, OverflowError):  # other number types, or numbers out of range
        if most is not None:
            values = np.minimum(values, most)
        numbers = np.empty(len(values), np.int64)
        numbers[:] = values
        return array("q", numbers.tolist())


class Sampler:
    """``forward`` takes float32 logits ``[R, V]`` and, per row, the request's
    parameters, its seed and the index of the draw (how many tokens the request has
    sampled before); it returns int32 tokens and float32 log-probabilities on the
    device.  NaN logits count as -1e5 (sampler.py:21-26)."""

    RING = 4  # pinned staging buffers in turn; one is reused only after its copy is done

    def __init__(self, device):
        self.device = torch.device(device)
        self._staging: list[tuple[torch.Tensor, torch.cuda.Event | None]] = []
        self._turn = 0

    def _stage(self, words: int) -> torch.Tensor:
        """A pinned int32 buffer of at least ``words`` entries whose last copy has finished."""
        if len(self._staging) < self.RING:
            self._staging.append((torch.empty(max(words, 1024), dtype=torch.int32, pin_memory=True), None))
            self._turn = len(self._staging) - 1
        else:
            self._turn = (self._turn + 1) % self.RING
        buf, event = self._staging[self._turn]
        if event is not None:
            event.synchronize()
        if buf.numel() < words:
            buf = torch.empty(2 * words, dtype=torch.int32, pin_memory=True)
        self._staging[self._turn] = (buf, None)
        return buf

    def forward(self, logits: torch.Tensor, params: list[SamplingParams], seeds: list[int], draw_index: list[int]):
        n = logits.shape[0]
        if not (len(params) == len(seeds) == len(draw_index) == n):
            raise ValueError("one parameter set, seed and draw index per row of logits")
        if n == 0:
            e = torch.empty(0, device=self.device)
            return e.to(torch.int32), e.to(torch.float32)
        # all per-row parameters in one buffer, one copy; a list a parameter, and the rest in one native call
        host = self._stage(7 * n)
        flags = ops.pack_sample_rows(
            host, array("d", [p.temperature for p in params]), array("d", [p.top_p for p in params]), array("d", [p.min_p for p in params]),
            _integers([p.top_k for p in params], 2**31 - 1), _integers(seeds), _integers(draw_index), logits.shape[1])
        dev = torch.empty(7 * n, dtype=torch.int32, device=self.device)
        dev.copy_(host[: 7 * n], non_blocking=True)
        event = torch.cuda.Event()
        event.record()
        self._staging[self._turn] = (host, event)
        return ops.sample_packed(logits.contiguous(), dev, flags)
