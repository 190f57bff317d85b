"""Which of the streaming tiles' loads pass the caches by, by the instructions that the compiler makes of them, without a GPU."""

import assembly


def test_weights_of_experts_pass_the_caches_by_where_a_group_has_one_tile():
    """A workgroup of experts decides it for its own group: the loop has a form of either kind, and rows of X are read from the caches in both."""
    kernels = {name: lines for name, lines in assembly.kernels("grouped_gemm.hip").items() if "grouped_stream_kernel" in name}
    experts = [lines for name, lines in kernels.items() if "grouped_stream_kernelILb0ELb1" not in name]
    assert len(kernels) == 3 and len(experts) == 2
    for name, lines in kernels.items():
        loads = [line for line in lines if line.startswith("buffer_load") and " lds" in line]
        once = sum(line.split()[-2:] == ["nt", "lds"] for line in loads)
        # (a step of tiles of 32 rows has one load of X and four of W, of 64 rows two and four)
        assert 2 * once > len(loads) * 0.6 and len(loads) - once > once if lines in experts else once == 0 and loads, name
