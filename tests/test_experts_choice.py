"""Which kernel takes experts of less than a row each where a round of the streaming tiles has just begun, by the times beside the rule, without a GPU."""

import pytest

from halite_amd.kernels import library

FEW, STREAM = 0, 1


# rows of up to 1,024 in the round's first fifth: the kernel for few rows; longer ones, and what lies outside the round: the streaming tiles
@pytest.mark.parametrize("n_rows, n, k, n_groups, gated, kernel", [
    (20, 4096, 1024, 64, False, FEW), (45, 2048, 512, 64, False, FEW), (40, 2048, 768, 256, False, FEW),
    (72, 512, 1536, 512, True, STREAM), (80, 512, 2048, 512, True, STREAM), (64, 768, 2048, 128, True, STREAM), (48, 1024, 4096, 64, True, STREAM),
    (30, 2048, 768, 256, False, STREAM), (60, 2048, 768, 256, False, STREAM), (64, 2048, 512, 64, False, STREAM)])
def test_a_round_begun(n_rows, n, k, n_groups, gated, kernel):
    assert library.core_library().hal_grouped_gemm_experts_kernel(n_rows, n, k, n_groups, int(gated)) == kernel
