"""Rotation and append of heads whose first columns still lie in another product's rows, against a copy of the columns first: the same bits."""

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 9, 1535, 1537])  # a token a workgroup, and eight
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("H, K, D, head, col, cols, rot, zero_from, n_zero, interleaved", [
    (4, 1, 96, 72, 40, 32, 32, 80, 16, False), (4, 1, 96, 72, 40, 32, 32, 80, 16, True), (3, 1, 64, 32, 0, 32, 16, 32, 0, False),  # some are not turned
    (5, 0, 64, 40, 8, 32, 0, 40, 24, False), (2, 1, 64, 48, 16, 32, 32, 56, 8, False),
    (4, 1, 96, 72, 36, 32, 32, 80, 16, False), (4, 1, 96, 72, 40, 20, 16, 84, 12, False),  # columns that are copied first: no whole pieces
])
def test_as_copied_first(gpu, n, dtype, H, K, D, head, col, cols, rot, zero_from, n_zero, interleaved):
    from halite_amd.kernels import ops

    gen = torch.Generator().manual_seed(n + D)
    rnd = lambda *s: torch.randn(s, generator=gen).to(dtype).to(gpu)  # noqa: E731
    x, rows = rnd(n, H * head + 8), rnd(n, (H + 2 * K) * D)
    page, table_len = 32, 400
    positions = (torch.arange(n, dtype=torch.int32) % 300 + 5).to(gpu)
    if n > 8 and rot:  # no position: the columns are there all the same, unturned
        positions[4], positions[n - 1] = -1, table_len
    seg = (torch.arange(n, dtype=torch.int32) // 300).to(gpu)
    n_seg = int(seg.max()) + 1
    table = torch.arange(n_seg * 10, dtype=torch.int32).view(n_seg, 10).to(gpu)
    angles = torch.rand((table_len, rot // 2), generator=gen) * 6
    cos, sin = angles.cos().to(gpu), angles.sin().to(gpu)
    got = []
    for together in (False, True):
        packed = rows.clone()
        pages = {}
        if K:
            pages = dict(token_seg=seg, block_table=table, page_size=page, tiled=D % 32 == 0 and dtype == torch.bfloat16,
                         k_pages=torch.zeros((n_seg * 10, K, page, D), dtype=dtype, device=gpu),
                         v_pages=torch.zeros((n_seg * 10, K, D, page), dtype=dtype, device=gpu))
        if not together:
            ops.head_cols(x, head, col, packed, D, 0, cols, H, zero_from=zero_from, n_zero=n_zero)
        ops.rope_append(packed, positions, cos, sin, H, K, D, rot, interleaved, **pages,
                        queries=ops.QueryColumns(x, head, col, cols, zero_from, n_zero) if together else None)
        got.append((packed, pages.get("k_pages"), pages.get("v_pages")))
    for a, b in zip(*got):
        assert a is None or torch.equal(a, b)
    assert not torch.equal(got[0][0], rows)


def test_what_is_refused(gpu):
    from halite_amd.kernels import ops

    rows, positions = torch.zeros((3, 64), device=gpu), torch.zeros(3, dtype=torch.int32, device=gpu)
    cos = torch.ones((4, 8), device=gpu)
    for x, head, col, cols, zeros in ((torch.zeros((2, 64), device=gpu), 32, 0, 16, (16, 0)), (torch.zeros((3, 32), device=gpu), 32, 0, 16, (16, 0)),
                                      (torch.zeros((3, 64), device=gpu), 32, 24, 16, (16, 0)), (torch.zeros((3, 64), device=gpu), 32, 0, 16, (24, 16))):
        with pytest.raises(ops.KernelError):
            ops.rope_append(rows, positions, cos, cos, 2, 0, 32, 16, False, queries=ops.QueryColumns(x, head, col, cols, *zeros))
