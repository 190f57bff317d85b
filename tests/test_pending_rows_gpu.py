"""What a layer leaves to be added up by the next reader is let go once it has been read: the rows of a mixture's experts are not
held beside those of the next mixture, nor beside the logits."""

import weakref

import pytest
import torch

import plain_kavuvik
import plain_vepitar
from halite_amd.config import ModelConfig, ServerConfig
from halite_amd.engine.batch import Segment
from halite_amd.engine.runner import ModelRunner

pytestmark = pytest.mark.gpu


def folder_of(model, tmp_path):
    if model.startswith("kavuvik"):
        P, cfg = plain_kavuvik, getattr(plain_kavuvik, "KAV_" + model[-1])
        weights = P.random_weights(cfg, seed=1)
    else:
        P, cfg = plain_vepitar, getattr(plain_vepitar, "VEP_" + model[-1])
        weights = P.random_weights(cfg, getattr(plain_vepitar, "VEP_" + model[-1] + "_RANKS"), seed=1)
    P.write_model_folder(str(tmp_path), cfg, weights, torch.bfloat16)
    return str(tmp_path)


@pytest.mark.parametrize("n_tokens", [1, 40])
@pytest.mark.parametrize("model", ["kavuvik A", "kavuvik B", "vepitar A", "vepitar B"])
def test_rows_are_let_go(gpu, model, n_tokens, tmp_path):
    server = ServerConfig(kv_cache_num_tokens=256, page_size=16, max_seqs_per_forward=4, use_cudagraph=False)
    runner = ModelRunner.from_pretrained(folder_of(model, tmp_path), server, ModelConfig(dtype="bfloat16"))
    left, at_head = [], []

    def held():
        return sum(r() is not None for r in left)

    for block in runner.model.layers.values():
        if hasattr(block.ff, "forward_sum"):
            def recorded(x, ctx, _f=block.ff.forward_sum):
                assert held() == 0
                s = _f(x, ctx)
                left.extend(weakref.ref(t) for t in (s.y, s.extra) if t is not None)
                return s

            block.ff.forward_sum = recorded
    head = runner.model.head.forward

    def recorded_head(x):
        at_head.append(held())
        return head(x)

    runner.model.head.forward = recorded_head
    slot = runner.admit()
    runner.step([Segment(slot, 0, list(range(1, n_tokens + 1)), [n_tokens - 1])])
    runner.free(slot)
    assert len(left) >= 2 and at_head == [0]
