"""Which of the streaming tiles' loads pass the caches by, by the instructions that the compiler makes of them, without a GPU."""

import assembly


def test_weights_of_experts_pass_the_caches_by_where_a_group_has_one_tile():
    """A workgroup of experts decides it for its own group: the loop has a form of either kind (of so few rows that all groups have one tile: one form),
    and rows of X are read from the caches in all."""
    kernels = {name: lines for name, lines in assembly.kernels("grouped_gemm.hip").items() if "grouped_stream_kernel" in name}
    assert len(kernels) == 5
    for name, lines in kernels.items():
        loads = [line for line in lines if line.startswith("buffer_load") and " lds" in line]
        once = sum(line.split()[-2:] == ["nt", "lds"] for line in loads)
        heads, one = "ILb0ELb1E" in name, "ELb0ELb1EE" in name
        # (a step of tiles of 32 rows has one load of X and four of W, of 64 rows two and four)
        share = 0.0 if heads else 8 / 11 if one else 8 / 22
        assert loads and abs(once / len(loads) - share) < 0.02, name
