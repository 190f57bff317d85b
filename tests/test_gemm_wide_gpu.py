"""The product of prompts in wide tiles against products in 64 bits: every height, edges of tiles in rows and columns, last rounds of
halved tiles, workgroups with several tiles, the shortest K, rows that lie apart, and the gates."""

from types import SimpleNamespace

import pytest
import torch
from test_grouped_wide_gpu import compare, rand

from halite_amd.kernels import library, ops
from halite_amd.parts.feedforward import GatedFeedForward

pytestmark = pytest.mark.gpu


@pytest.fixture
def gpu():
    return torch.device("cuda:0")


def check(gpu, m, n, k, height, out_dtype, apart=0):
    x, w = rand(m, k + apart, seed=m, scale=1.0).bfloat16().to(gpu)[:, :k], rand(n, k + apart, seed=n, scale=0.1).bfloat16().to(gpu)[:, :k]
    y = ops.gemm_bf16_wide(x, w, out_dtype=out_dtype, height=height)
    xs, ws = x.double(), w.double()
    compare(y, xs @ ws.T, (k, xs.abs() @ ws.abs().T), 2.0**-8 if out_dtype == torch.bfloat16 else 0.0)


# rows: one, the ends of blocks, octets and halves, a tile and one row more, several; columns: the fewest, inside a lane's eight, a
# wave's and a tile's end
@pytest.mark.parametrize("height", range(4, 12))
@pytest.mark.parametrize("out_dtype", [torch.bfloat16, torch.float32])
def test_tiles_of_every_height(gpu, height, out_dtype):
    r = 32 * height
    for m, n, k, apart in [(1, 4, 128, 0), (r - 1, 256, 256, 8), (r, 260, 128, 0), (r + 1, 516, 384, 0), (r // 2 + 9, 28, 128, 8), (2 * r + r // 2, 1028, 256, 0)]:
        check(gpu, m, n, k, height, out_dtype, apart)


# tiles over the 8 dies of 32 units: fewer than a round, half a round and one more, several rounds, a rest of halves beside them
@pytest.mark.parametrize("m, n, k, height", [(1000, 4096, 128, 4), (2048, 4224, 128, 8), (2048, 4352, 256, 8), (4100, 8192, 128, 4), (3000, 8448, 128, 5),
                                             (2816, 16640, 128, 11), (3201, 14336, 128, 10), (4500, 4864, 128, 0), (700, 20608, 128, 0)])
def test_rounds_and_their_rests(gpu, m, n, k, height):
    check(gpu, m, n, k, height, torch.float32)
    check(gpu, m, n, k, height, torch.bfloat16)


@pytest.mark.parametrize("activation, clamp", [("silu", ops.Clamp()), ("gelu_tanh", ops.Clamp()), ("clamped", ops.Clamp(1.5, 1.702, 1.0))])
@pytest.mark.parametrize("m, n, k, height", [(1, 128, 128, 4), (300, 132, 256, 5), (2048, 2304, 128, 8), (353, 1300, 384, 11), (1500, 4096, 128, 0), (2200, 11008, 128, 7)])
def test_gated(gpu, m, n, k, height, activation, clamp):
    x = rand(m, k, seed=m).bfloat16().to(gpu)
    both = rand(2 * n, k, seed=n, scale=0.15).bfloat16().to(gpu)
    y = ops.gemm_bf16_wide(x, both[:n], w_up=both[n:], activation=activation, clamp=clamp, height=height)
    xs, ws = x.double(), both.double()
    g, u = xs @ ws[:n].T, xs @ ws[n:].T
    off_g, off_u = ((k + 8) * 2.0**-23 * (xs.abs() @ w.abs().T) for w in (ws[:n], ws[n:]))
    if activation == "clamped":
        g, u = g.clamp(max=clamp.limit), u.clamp(-clamp.limit, clamp.limit) + clamp.up_shift
        a = g * torch.sigmoid(clamp.alpha * g)
    else:
        a = torch.nn.functional.silu(g) if activation == "silu" else torch.nn.functional.gelu(g, approximate="tanh")
    want = a * u
    # an activation's slope is at most 1.2; its sigmoid is off by the exponential's argument, |z| 2^-23, and a few roundings
    limit = 1.2 * off_g * u.abs() + off_u * a.abs() + (2.0**-8 + (4 + 4 * g.abs()) * 2.0**-22) * want.abs() + 1e-30
    assert bool(((y.double() - want).abs() <= limit).all()), float(((y.double() - want).abs() / limit).max())


def test_what_is_not_finite_stays_so(gpu):
    x, w = rand(200, 128, seed=1).bfloat16().to(gpu), rand(2 * 128, 128, seed=2).bfloat16().to(gpu)
    x[3, 5], x[7, 9] = float("nan"), float("inf")
    y = ops.gemm_bf16_wide(x, w, out_dtype=torch.float32)
    want = x.float() @ w.float().T
    assert torch.equal(torch.isfinite(y), torch.isfinite(want)) and bool(torch.isnan(y[3]).all())
    act = ops.gemm_bf16_wide(x, w[:128], w_up=w[128:])
    assert bool(torch.isnan(act[3]).all()) and bool(torch.isfinite(act[8:]).all())


def test_a_row_does_not_depend_on_its_neighbours(gpu):
    x, w = rand(1500, 256, seed=7).bfloat16().to(gpu), rand(1024, 256, seed=8).bfloat16().to(gpu)
    whole = ops.gemm_bf16_wide(x, w, height=4)
    for height in (5, 8, 11):
        assert torch.equal(whole, ops.gemm_bf16_wide(x, w, height=height))
    assert torch.equal(whole[77:300], ops.gemm_bf16_wide(x[77:300], w))


def test_what_linear_takes(gpu):
    """Where the rule says so, ``linear`` goes to the wide tiles; sizes and places that they do not have stay where they were."""
    lib = library.core_library()
    assert lib.hal_gemm_bf16_wide_pays(2048, 4096, 4096, 0, 0) and lib.hal_gemm_bf16_wide_pays(2048, 14336, 4096, 1, 0)
    assert not lib.hal_gemm_bf16_wide_pays(8192, 4096, 4096, 0, 0) and not lib.hal_gemm_bf16_wide_pays(64, 14336, 4096, 1, 0)
    x = rand(2048, 2056, seed=1).bfloat16().to(gpu)
    w = rand(2048, 2056, seed=2, scale=0.1).bfloat16().to(gpu)
    assert ops.wide_pays(x[:, :2048], w[:, :2048], 2048)
    for a, b in [(x[:, :2048], w[:, :2048]), (x[:, 4:2052], w[:, 4:2052]), (x, w), (x[:, :2000], w[:, :2000])]:
        if b.shape[1] != 2048 or b.storage_offset():
            assert not ops.wide_pays(a, b, 2048)
        for dtype in (torch.bfloat16, torch.float32):
            y, xs, ws = ops.linear(a, b, out_dtype=dtype), a.double(), b.double()
            assert not ops.wide_pays(a, b, 2048, out_dtype=dtype) or torch.equal(y, ops.gemm_bf16_wide(a, b, out_dtype=dtype))
            compare(y, xs @ ws.T, (b.shape[1], xs.abs() @ ws.abs().T), 2.0**-8 if dtype == torch.bfloat16 else 0.0)


@pytest.mark.parametrize("f, wide", [(2048, True), (2056, False)])
def test_what_the_gated_form_takes(gpu, monkeypatch, f, wide):
    """The feed-forward's gated product goes to the wide tiles where the rule says so, and to the product and its gate's kernel where it does not."""
    x, both, down = rand(2048, 512, seed=1), rand(2 * f, 512, seed=2, scale=0.1), rand(512, f, seed=3, scale=0.1)
    x, both, down = (t.bfloat16().to(gpu) for t in (x, both, down))
    took, real = [], ops.gemm_bf16_wide
    monkeypatch.setattr(ops, "gemm_bf16_wide", lambda *a, **k: took.append("w_up" in k) or real(*a, **k))
    if not wide:
        monkeypatch.setattr(ops, "_wide_pays", lambda *a: False)
    part = SimpleNamespace(p=SimpleNamespace(intermediate_size=f, float32_result=False), w_gate_up=both, w_out=down, t_gate=None, t_out=None)
    y = GatedFeedForward.forward(part, x, None)
    assert (True in took) == wide
    act = torch.nn.functional.silu(x.double() @ both[:f].double().T) * (x.double() @ both[f:].double().T)
    # act is rounded once or (in two kernels) three times to 8 bits, its error and the result's rounding
    limit = 4 * 2.0**-8 * (act.abs() @ down.double().abs().T)
    assert bool(((y.double() - act @ down.double().T).abs() <= limit).all())
