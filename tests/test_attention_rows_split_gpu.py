"""Float32 attention of prompts: waves that share the rows and split the keys where a step has up to 256 workgroups, and
waves that have their rows to themselves where it has more."""

import pytest
import torch
from test_kernels_gpu import attention_case

pytestmark = pytest.mark.gpu


# 32 tokens a workgroup times 8 heads of keys: 256 workgroups and 264 (and 304 of 128 tokens); several requests in one workgroup; portions
@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("H, K, D, segs", [(32, 8, 128, [(0, 1024)]), (32, 8, 128, [(0, 1025)]), (32, 8, 96, [(70, 1060)]), (16, 16, 64, 9 * [(0, 260)]),
                                           (32, 8, 72, [(0, 33), (31, 34), (63, 9), (64, 130), (500, 40)]), (12, 4, 128, [(0, 300), (129, 31)])])
def test_split_and_whole(dtype, H, K, D, segs):
    for page, window in ((16, 0), (64, 37)):
        attention_case(torch.device("cuda:0"), dtype, H, K, D, page, segs, window, seed=31, use="simple")
