"""When a step's long segments go to the attention kernel for long segments: values that are read in all
dimensions need a workgroup a compute unit wherever the zeros that a layer declares are not left out, and
chunks bound the keys that a row sees."""

import pytest

from halite_amd.kernels import attention as attn_kernels


@pytest.mark.parametrize("head_dim, value_from, skipped", [(256, 64, True), (256, 128, True), (256, 48, False), (160, 64, False), (160, 0, False)])
def test_zeros_left_out(head_dim, value_from, skipped):
    assert bool(attn_kernels.skips_leading_zeros(head_dim, value_from)) == skipped
    # 1,024 tokens of 16 heads over one: 128 workgroups, 8.4 million (row, key) pairs; of 32 heads 256 workgroups
    pay = attn_kernels.long_items_pay
    assert pay([1024], [1024], 16, 1, 0, head_dim, value_from) == skipped
    assert pay([1024], [1024], 32, 1, 0, head_dim, value_from)


def test_chunks_bound_the_keys():
    pay = attn_kernels.long_items_pay
    assert pay([64], [4160], 32, 1, 0, 256, 64) and not pay([64], [4160], 32, 1, 0, 256, 64, 100)
    assert pay([4096], [4096], 4, 4, 0, 160, 0, 256) and not pay([4096], [4096], 4, 4, 0, 160, 0, 80)
