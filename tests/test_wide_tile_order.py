"""Reads of LDS in the wide tiles, by the instructions that the compiler makes of them, without a GPU: what a wave reads in a phase has come
before the phase's last barrier.  The other group of waves asks for that place anew behind it, without a wait of its own for these reads."""

import re
from concurrent.futures import ThreadPoolExecutor

import assembly

KERNELS = {"gemm_wide.hip": "gemm_wide_kernel", "grouped_gemm.hip": "grouped_wide_kernel"}


def late(lines):
    """The reads that may be on their way over a second barrier: (line, line of the barrier)."""
    reads, found = [], []  # of a read not waited for: its line, barriers since
    for at, line in enumerate(lines):
        if line.startswith("ds_read"):
            reads.append([at, 0])
        elif line.startswith("s_waitcnt") and (m := re.search(r"lgkmcnt\((\d+)\)", line)):
            reads = reads[max(0, len(reads) - int(m[1])):]  # (LDS answers in order)
        elif line.startswith("s_barrier"):
            for read in reads:
                read[1] += 1
            found += [(read[0], at) for read in reads if read[1] == 2]
    return found


def test_a_phase_has_its_operands_before_it_ends():
    with ThreadPoolExecutor() as pool:
        bodies = {name: lines for source, found in zip(KERNELS, pool.map(assembly.kernels, KERNELS)) for name, lines in found.items() if KERNELS[source] in name}
    assert len(bodies) == 34  # eight heights, plain and gated, read once or not; two of the experts'
    for name, lines in bodies.items():
        assert sum(line.startswith("s_barrier") for line in lines) >= 16 and sum(line.startswith("v_mfma") for line in lines) >= 64, name
        assert not late(lines), (name, [(lines[a], lines[b]) for a, b in late(lines)[:4]])


def test_the_reading_itself():
    barrier, read = "s_barrier", "ds_read_b128 v[0:3], v4"
    assert not late([read, barrier, "s_waitcnt lgkmcnt(0)", barrier])
    assert late([read, read, barrier, "s_waitcnt vmcnt(3)", barrier]) == [(0, 4), (1, 4)]
    assert late([read, read, barrier, "s_waitcnt lgkmcnt(1)", barrier]) == [(1, 4)]
