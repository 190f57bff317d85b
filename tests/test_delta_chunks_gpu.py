"""The generalized delta rule in chunks of 16 tokens (``ops.delta_chunks``) against the plain recurrence in 64 bits:
segments around a chunk's and a group of segments' edges, ranks around the 64 that are held at a time, heads that
do not fill a workgroup, states that are not zero, rows of other slots untouched; what an infinite value reaches; and
which calls the rule takes to it."""

import math

import pytest
import torch

import plain_vepitar as P
from halite_amd.kernels import ops

pytestmark = pytest.mark.gpu
F = torch.float64
D = 64
RATE, UNIT_EPS, EPS = math.exp(-0.5), 1e-6, 1e-5


def rand(*shape, seed=0, scale=1.0):
    return scale * torch.randn(*shape, generator=torch.Generator().manual_seed(seed))


def inputs(gpu, H, rank, lens, stored=torch.float32, seed=1):
    n, T, S = H * D, sum(lens), len(lens)
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device=gpu)  # noqa: E731
    a = rand(T, 5 * n + -(-rank // 4) * 4, seed=seed)
    w2, w0, ab = rand(n, rank, seed=seed + 1, scale=0.8 / max(1.0, rank / 8) ** 0.5).to(stored), rand(n, seed=seed + 2).to(stored), rand(n, seed=seed + 3).to(stored)
    weight = rand(n, seed=seed + 4).to(stored)
    state = torch.full((S + 2, H, D, D), float("nan"))
    state[1 : S + 1] = 0.3 * rand(S, H, D, D, seed=seed + 5)
    slots = [S - i for i in range(S)]  # the last request lives in the first slot that is used
    return dict(a=a, w2=w2, w0=w0, ab=ab, weight=weight, state=state, slots=slots, lens=lens, H=H, rank=rank,
                starts=i32([sum(lens[:i]) for i in range(S)]), counts=i32(lens), slot=i32([s for s, m in zip(slots, lens) for _ in range(m)]))


def run(gpu, x, dtype=torch.float32, rate=RATE):
    a, n = x["a"].to(gpu), x["H"] * D
    r, k, v, a_raw, z = (a[:, i * n : (i + 1) * n] for i in range(5))
    state = x["state"].clone().to(gpu)
    y = ops.delta_chunks(r, k, v, a_raw, a[:, 5 * n : 5 * n + x["rank"]], x["w2"].to(gpu), x["w0"].to(gpu), x["ab"].to(gpu), state,
                         x["starts"], x["counts"], x["slot"], rate, UNIT_EPS, z, x["weight"].to(gpu), EPS, dtype)
    return y.cpu(), state.cpu()


def plain(x, segment, rate=RATE):
    """The segment's rows and the state after it, in 64 bits."""
    H, n = x["H"], x["H"] * D
    t0 = sum(x["lens"][:segment])
    b = x["a"][t0 : t0 + x["lens"][segment]].to(F)
    r, k, v, a_raw, z = (b[:, i * n : (i + 1) * n].view(-1, H, D) for i in range(5))
    decay = torch.exp(-rate * torch.sigmoid(torch.tanh(b[:, 5 * n : 5 * n + x["rank"]]) @ x["w2"].to(F).T + x["w0"].to(F))).view(-1, H, D)
    rate = torch.sigmoid(a_raw + x["ab"].to(F).view(H, D))
    start = x["state"][x["slots"][segment]].to(F)
    heads = [P.delta_recurrence(r[:, h], k[:, h], v[:, h], decay[:, h], rate[:, h], start[h]) for h in range(H)]
    o = torch.stack([o for o, _ in heads], 1)
    y = o / torch.sqrt((o * o).mean(-1, keepdim=True) + EPS) * x["weight"].to(F).view(H, D) * torch.sigmoid(z)
    return y.reshape(-1, n), torch.stack([s for _, s in heads])


@pytest.mark.parametrize("H,rank,lens,stored", [
    (1, 1, [1, 2], "float32"), (3, 5, [15, 16, 17], "bfloat16"), (4, 63, [33, 1, 64, 3], "float32"), (5, 64, [48, 31], "bfloat16"),
    (2, 66, [130], "bfloat16"), (2, 132, [5, 80], "float32"), (1, 8, [1 + i % 19 for i in range(130)], "float32")])
def test_rows_and_states(gpu, H, rank, lens, stored):
    """A chunk's sums are as long as the walk's, so the bound is that of the other delta-rule tests: 3e-5 of the largest number."""
    x = inputs(gpu, H, rank, lens, stored=getattr(torch, stored))
    y, state = run(gpu, x)
    for i in sorted({0, 1, len(lens) // 2, 63, 64, len(lens) - 1} & set(range(len(lens)))):
        want, left = plain(x, i)
        t0 = sum(lens[:i])
        assert float((y[t0 : t0 + lens[i]] - want).abs().max()) < 3e-5 * max(1.0, float(want.abs().max())), (i, lens[i])
        assert float((state[x["slots"][i]] - left).abs().max()) < 3e-5 * max(1.0, float(left.abs().max())), (i, lens[i])
    assert bool(torch.isnan(state[0]).all()) and bool(torch.isnan(state[-1]).all())
    rounded, _ = run(gpu, x, torch.bfloat16)
    assert torch.equal(rounded, y.to(torch.bfloat16))


@pytest.mark.parametrize("rate", [1e-4, 1.5, 2.5])
@pytest.mark.parametrize("bias", ["strong", "weak", "mixed"])
def test_rates_up_to_the_largest(gpu, rate, bias):
    """Decays near exp(-rate) in every token (a chunk's product is then exp(-16 rate), 4e-18 at the largest rate, which keys are
    divided by), near 1, and both among a head's channels; the bound is that of the rows and states above."""
    H, lens = 3, [16, 47, 33]
    x = inputs(gpu, H, 8, lens, seed=9)
    shift = torch.full((H * D,), 12.0)
    if bias != "strong":
        shift[(torch.arange(H * D) % 2 == 0) | (bias == "weak")] = -12.0
    x["w0"] = x["w0"] + shift
    y, state = run(gpu, x, rate=rate)
    for i in range(len(lens)):
        want, left = plain(x, i, rate)
        t0 = sum(lens[:i])
        assert float((y[t0 : t0 + lens[i]] - want).abs().max()) < 3e-5 * max(1.0, float(want.abs().max())), (i, lens[i])
        assert float((state[x["slots"][i]] - left).abs().max()) < 3e-5 * max(1.0, float(left.abs().max())), (i, lens[i])


@pytest.mark.parametrize("stored", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("off", [1, 2, 3])
def test_weights_that_begin_inside_a_vector(gpu, off, stored):
    x = inputs(gpu, 3, 8, [33, 16], stored=stored)
    moved = dict(x, **{name: torch.cat((x[name].new_zeros(off), x[name].flatten())).to(gpu)[off:].view(x[name].shape) for name in ("w2", "w0", "ab", "weight")})
    assert moved["w2"].data_ptr() % (4 * moved["w2"].element_size()) != 0 and moved["weight"].data_ptr() % (4 * moved["weight"].element_size()) != 0
    (y, state), (y2, state2) = run(gpu, x), run(gpu, moved)
    assert torch.equal(y, y2) and torch.equal(state[1:-1], state2[1:-1])


@pytest.mark.parametrize("what", [0, 1, 2, 3, 4])  # r, k, v, a, z
@pytest.mark.parametrize("value", [float("inf"), float("nan")])
def test_an_infinite_number_reaches_no_token_before_it(gpu, what, value):
    H, lens = 2, [37, 20]
    x = inputs(gpu, H, 8, lens, seed=7)
    clean, clean_state = run(gpu, x)
    at, channel = 21, 70  # of the first request, in its second chunk; a channel of the second head
    x["a"][at, what * H * D + channel] = value
    y, state = run(gpu, x)
    assert torch.equal(y[:at], clean[:at]) and torch.equal(y[lens[0] :], clean[lens[0] :])
    assert torch.equal(y[:, :D], clean[:, :D])  # (the other head)
    assert torch.equal(state[x["slots"][1]], clean_state[x["slots"][1]])
    touched = y[at : lens[0], D:]
    if what == 2:  # a value: its channel of every later row and of the state, and with it the norm of the head
        assert not bool(torch.isfinite(touched[:, channel - D]).any())
        assert not bool(torch.isfinite(state[x["slots"][0]][1][:, channel - D]).any())


def test_which_calls_the_rule_takes(gpu):
    rows = torch.zeros((64, 4 * 64 + 4), device=gpu)
    v, z = rows[:, :256], rows[:, 4:]
    fit = lambda v=v, z=z, n=4, heads=4, dim=64, rate=RATE: ops.delta_chunks_fit(v, z, n, heads, dim, rate)  # noqa: E731
    assert fit() and fit(n=64, heads=8)
    assert not fit(n=16, heads=64) and fit(n=8, heads=128)  # chunks mostly empty, many of them; filled ones
    assert not fit(dim=128) and not fit(rate=2.6)  # other heads; decays so strong that their products vanish
    assert not fit(v=rows[:, 1:257]) and not fit(z=rows[:, 2:258])  # rows off 16 bytes
    odd = torch.zeros((64, 4 * 64 + 3), device=gpu)
    assert not fit(v=odd[:, :256])
