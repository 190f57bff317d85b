"""Float32 products of prompts by parts of bf16: edges of tiles, parts of K, rows in turns, and numbers that have no parts."""

import pytest
import torch

from halite_amd.kernels import library, ops


def _operands(m, n, k):
    gen = torch.Generator().manual_seed(m + n + k)
    return torch.randn(m, k, generator=gen).cuda(), (torch.randn(n, k, generator=gen) * 0.02).cuda()


# the fewest rows, a tile of each height and one row more; one part of K to eight, of unequal lengths, an odd number of stages in
# a part, K that ends inside a stage; columns that end inside a tile and inside a vector; rows in two turns over their planes
@pytest.mark.gpu
@pytest.mark.parametrize("m, n, k", [(65, 96, 2048), (128, 130, 2052), (96, 12300, 2056), (129, 4090, 2080), (257, 6147, 2116), (300, 8200, 2048),
                                     (513, 16388, 2084), (1100, 3072, 2048), (1025, 4097, 4100), (200, 1000, 14336),
                                     (66, 8300, 4132), (129, 8201, 4100), (400, 8196, 8260)])  # the last three: totals in turns
def test_sizes(m, n, k):
    a, w = _operands(m, n, k)
    lib = library.core_library()
    assert lib.hal_gemm_f32_split_takes(ops._ptr(a), k, ops._ptr(w), k, m, k)
    w[n // 2] = w[n // 2].abs()  # (sums without cancellation: of a stretch left out, doubled or rounded to one side)
    a[m // 2] = a[m // 2].abs()
    got = ops.gemm_f32(a, w)
    want, size = a.double() @ w.double().T, a.double().abs() @ w.double().abs().T
    # a float32 addition a stage of 32; in a stage six sums that are cut off and the products left out: at most 2 and 1 each
    assert bool(((got.double() - want).abs() <= (k // 32 + 16) * 2.0**-24 * size).all())
    # a row's result is its own, whatever tile it is in and whatever rows are beside it
    assert torch.equal(ops.gemm_f32(a[: m - 1].contiguous(), w) if m > 65 else got[:-1], got[: m - 1])
    if m > 200:
        assert torch.equal(ops.gemm_f32(a[m - 70 :].contiguous(), w), got[m - 70 :])


@pytest.mark.gpu
@pytest.mark.parametrize("m, n, k", [(130, 300, 2052), (300, 8200, 2048), (130, 8201, 4132)])
def test_numbers_without_parts(m, n, k):
    a, w = _operands(m, n, k)
    inf, nan, most = float("inf"), float("nan"), 3.4e38  # (the last: a float32 number that rounds to a bf16 infinity)
    w[:, 40] = 1e-30
    a[3, 5], a[4, 7], a[4, 2047], a[100, 9], a[128, 40], a[129, 0] = inf, inf, -inf, nan, most, most
    w[17, 11], w[n - 1, 2], w[18, 700] = -inf, nan, inf
    a[7, 700] = 0.0
    got = ops.gemm_f32(a, w)
    want = a.double() @ w.double().T
    want = torch.where(want.abs() > 3.4028235e38, want.sign() * inf, want)
    assert torch.equal(got.isnan(), want.isnan())
    finite = want.isfinite()
    assert torch.equal(got[~finite & ~want.isnan()].double(), want[~finite & ~want.isnan()])
    plain = a.nan_to_num(0, 0, 0).double().abs() @ w.nan_to_num(0, 0, 0).double().abs().T
    assert bool(((got.double() - want).abs() <= (k // 32 + 16) * 2.0**-24 * plain)[finite].all())
    # columns of W that begin off a vector go to the other tiles
    off = torch.empty(n * k + 1, device="cuda")[1:].view(n, k).copy_(w)
    assert not library.core_library().hal_gemm_f32_split_takes(ops._ptr(a), k, ops._ptr(off), k, m, k)
    assert torch.equal(ops.gemm_f32(a, off).isnan(), got.isnan())


# ---- as exact as float32 sums: what no bound on a sum's largest error can tell ----------------------------------------------
# Each of the six products that are added up, the bound that the tests below set on the error's norm over the result's, and
# operands whose parts have one sign, so that a product left out or paired wrongly cannot cancel.
SIX = [(0, 0), (0, 1), (1, 0), (0, 2), (2, 0), (1, 1)]  # parts of A and W (0: high, 1: middle, 2: low)


def _parts_of_one_sign(m, n, k, gen):
    """Numbers whose three parts are all positive: (128 + i) / 128 + j 2^-16 + l 2^-23, which float32 holds and whose last two
    are under half of the first one's unit together; A's middle and low parts are near their largest, W's are smaller, so
    that no two of the products are alike."""
    def numbers(rows, middle, low):
        i, j, l = (torch.randint(*between, (rows, k), generator=gen) for between in ((0, 128), middle, low))
        return (((128 + i) * 2**16 + j * 2**7 + l).double() * 2.0**-23).float()

    return numbers(m, (200, 255), (40, 64)), numbers(n, (128, 160), (10, 20))


def _by_parts(a, w, which, scale=2.0**16):
    """The sum in 64 bits of chosen products of the parts."""
    def parts(x):
        out, x = [], x.double() * scale
        for _ in range(3):
            out.append(x.float().bfloat16().double())
            x = x - out[-1]
        return out

    pa, pw = parts(a), parts(w)
    return sum(pa[i] @ pw[j].T for i, j in which) / scale**2


def _off(got, want):
    return float((got.double() - want).norm() / want.norm())


# what the six products leave out is under 2^-24 of each product; a sum's float32 additions lose 1.5e-7 (see the kernel)
ONE_SIGN_BOUND = 2.0**-24 + 1.5e-7


@pytest.mark.parametrize("k", [2048, 4096])
def test_the_bound_tells_each_product(k):
    """On the CPU: all six products are far inside of the bounds, and with any one left out, or in the place of another, outside."""
    gen = torch.Generator().manual_seed(k)
    a, w = _parts_of_one_sign(6, 5, k, gen)
    want = a.double() @ w.double().T
    assert _off(_by_parts(a, w, SIX), want) < 2.0**-24
    for left in SIX:
        rest = [p for p in SIX if p != left]
        assert _off(_by_parts(a, w, rest), want) > 3 * ONE_SIGN_BOUND
        for other in rest:
            assert _off(_by_parts(a, w, rest + [other]), want) > 3 * ONE_SIGN_BOUND
    # and of ordinary numbers the low parts: more than ten times what float32 sums lose
    a, w = torch.randn(6, k, generator=gen), torch.randn(5, k, generator=gen) * 0.02
    want = a.double() @ w.double().T
    assert _off(_by_parts(a, w, SIX), want) < 1e-7
    for rest in (SIX[:3] + SIX[5:], SIX[:4] + SIX[5:], SIX[:3] + SIX[4:]):
        assert _off(_by_parts(a, w, rest), want) > 1e-6


@pytest.mark.parametrize("e_a, e_w", [(0, 0), (-125, 0), (0, -120), (-120, 100), (-100, -20)])
def test_no_bit_of_a_small_number_is_lost(e_a, e_w):
    """On the CPU: the parts of scaled numbers hold all bits down to float32's smallest."""
    gen = torch.Generator().manual_seed(1)
    a, w = torch.randn(6, 2048, generator=gen) * 2.0**e_a, torch.randn(5, 2048, generator=gen) * 2.0**e_w
    all_nine = [(i, j) for i in range(3) for j in range(3)]
    assert _off(_by_parts(a, w, all_nine), a.double() @ w.double().T) < 1e-15


# (each in one part, several, several walks; the number of rows takes tiles of each height)
EXACT_SIZES = [(65, 96, 2048), (128, 4096, 4096), (130, 16500, 4100), (300, 6144, 4096), (520, 8200, 2084), (70, 8300, 8192), (200, 8192, 14336), (80, 4096, 14336)]


@pytest.mark.gpu
@pytest.mark.parametrize("m, n, k", EXACT_SIZES)
def test_every_product_of_parts_is_there(m, n, k):
    gen = torch.Generator().manual_seed(m)
    a, w = (x.cuda() for x in _parts_of_one_sign(m, n, k, gen))
    want = a.double() @ w.double().T
    off = (ops.gemm_f32(a, w).double() - want) / want
    assert float(off.norm() / off.numel() ** 0.5) < ONE_SIGN_BOUND
    # and in every row and column
    assert float(off.square().mean(0).sqrt().max()) < 2 * ONE_SIGN_BOUND and float(off.square().mean(1).sqrt().max()) < 2 * ONE_SIGN_BOUND


@pytest.mark.gpu
@pytest.mark.parametrize("kind", ["of both signs", "without signs", "beside one", "wide"])
@pytest.mark.parametrize("m, n, k", EXACT_SIZES)
def test_as_exact_as_the_float32_instruction(m, n, k, kind):
    """The distance to 64 bits is no larger than that of the product in float32 multiply-adds."""
    a, w = _operands(m, n, k)
    if kind == "without signs":
        a, w = a.abs(), w.abs()
    elif kind == "beside one":
        a, w = a + 1.0, w + 0.01
    elif kind == "wide":
        a = a * torch.exp(2.0 * torch.randn(a.shape, generator=torch.Generator().manual_seed(9))).cuda()
    lib, before = library.core_library(), torch.empty((m, n), device="cuda")
    assert lib.hal_gemm_f32(ops._ptr(a), k, ops._ptr(w), k, ops._ptr(before), n, m, n, k, ops._stream()) == 0
    want = a.double() @ w.double().T
    assert _off(ops.gemm_f32(a, w), want) <= _off(before, want) < 2e-6


@pytest.mark.gpu
@pytest.mark.parametrize("e_a, e_w", [(-104, 0), (-116, 0), (-125, 0), (0, -120), (-116, 100), (-60, -50), (100, -100), (108, -20), (113, -40)])
def test_small_and_large_numbers_keep_their_bits(e_a, e_w):
    """Below 2^-109 a number's low part would fall under bf16's smallest; from 2^112 on, results are taken as float32 sums."""
    a, w = _operands(130, 300, 2052)
    a, w = a * 2.0**e_a, (w * 64.0) * 2.0**e_w
    want = a.double() @ w.double().T
    assert float(want.abs().min()) > 2.0**-126 * 2.0**-20 and _off(ops.gemm_f32(a, w), want) < 4e-7
