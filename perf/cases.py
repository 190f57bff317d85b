"""What the engine's speed is measured on: serving work through its public entry points.

``listed`` names the cases, ``draw`` gives further ones of the same ranges, ``prepare`` builds what
a program holds before the call (a model with weights, its cache, the requests), ``run`` is one
pass, ``work`` what a pass cannot do without, ``exact`` the same results in 64 bits.

A case is one of five kinds:

* ``decode``: one step of ``ModelRunner.step`` with a token of each of ``requests`` live requests
  whose contexts are filled beforehand (every pass is one position on, as in serving), from a
  captured graph;
* ``prefill``: the prompts of ``requests`` new requests, admitted, fed in steps of at most
  ``portion`` tokens, the logits of every prompt's last token, and freed;
* ``score``: the same with the logits of every token wanted (what ``bin/trace_run`` does);
* ``serve``: ``InferenceEngine.infer_batch``: a batch of requests from token ids to generated
  tokens and their log-probabilities, greedy, prompts in portions beside decoded tokens;
* ``sample``: ``Sampler.forward`` on a step's logits, with temperature and top-p.

The models are layers of the shapes that ``bench.py`` serves (Llama-3.1-8B and Llama-3.2-3B
shapes, Kavuvik and Vepitar at its two sizes) with random weights; fewer layers than the whole
model where a pass does not depend on their number, which keeps inputs quick to make.
Embeddings stand out from what the layers add to them and routers prefer some experts by token,
as in trained mixtures: a rounding then does not turn over a choice between two experts of equal score.
"""

from __future__ import annotations

import math
import random

import numpy as np
import torch

from halite_amd.config import ModelConfig, ServerConfig, parse_config
from halite_amd.engine import InferenceEngine, ModelRunner, Segment
from halite_amd.sampling import Sampler, SamplingParams

DEVICE = "cuda"
PAGE = 64
F64 = torch.float64
LONGEST_STEP = 8192  # tokens of a prompt step
EXACT_FLOPS = 6.0e14  # what ``exact`` takes on at most (some 15 seconds in 64 bits)

LLAMA = {
    "llama-8b": dict(width=4096, heads=32, kv_heads=8, dim=128, ff=14336, factor=8.0),
    "llama-3b": dict(width=3072, heads=24, kv_heads=8, dim=128, ff=8192, factor=32.0),
}
KAVUVIK = {
    "kavuvik-2048": dict(width=2048, heads=16, dim=128, rot_dim=64, vdim=128, q_rank=768, kv_rank=192,
                         experts=32, top=4, ff=512, shared_ff=1024),
    "kavuvik-4096": dict(width=4096, heads=32, dim=128, rot_dim=64, vdim=128, q_rank=1536, kv_rank=192,
                         experts=64, top=6, ff=1024, shared_ff=2048),
}
VEPITAR = {
    "vepitar-2048": dict(width=2048, heads=16, kv_heads=4, dim=128, window=1024, conv=4, delta_heads=32, delta_dim=64,
                         decay_rank=64, experts=16, top=4, expert_ff=2048, dense_ff=5504, streams=2),
    "vepitar-4096": dict(width=4096, heads=32, kv_heads=8, dim=128, window=1024, conv=4, delta_heads=64, delta_dim=64,
                         decay_rank=64, experts=16, top=4, expert_ff=4096, dense_ff=11008, streams=2),
}
KAVUVIK_LIMIT, KAVUVIK_ALPHA = 7.0, 1.702
RESIDUAL_MULT = 0.5
ROUTING_STRENGTH = 8.0  # how far a token's embedding reaches along its experts' directions, in standard deviations


def listed():
    bf16 = dict(dtype="bfloat16")
    llama8 = dict(model="llama-8b", layers=8, vocab=128256)
    kavuvik = dict(model="kavuvik-4096", layers=4, vocab=32000)
    vepitar = dict(model="vepitar-4096", layers=4, vocab=32000)
    return [
        # one user's reply: latency of a token, where launches and small reads count
        dict(name="llama decode 1", kind="decode", requests=1, context=512, ragged=False, **llama8, **bf16),
        # long documents: weights and the cache weigh alike
        dict(name="llama decode 8 long", kind="decode", requests=8, context=8192, ragged=False, **llama8, **bf16),
        # a busy server: many chats of different lengths
        dict(name="llama decode 64", kind="decode", requests=64, context=1100, ragged=True, **llama8, **bf16),
        # the time to the first token of an ordinary prompt
        dict(name="llama prefill 2048", kind="prefill", requests=1, context=2048, ragged=False, portion=8192, **llama8, **bf16),
        # a long prompt in one step: attention begins to count
        dict(name="llama prefill 8192", kind="prefill", requests=1, context=8192, ragged=False, portion=8192, **llama8, **bf16),
        # a whole batch through the scheduler: portions beside decoded tokens, sampling, results on the host
        dict(name="llama serve 16", kind="serve", requests=16, context=2000, ragged=True, portion=512, new=48,
             model="llama-3b", layers=8, vocab=128256, **bf16),
        # scoring a text on the exactness path
        dict(name="llama score float32", kind="score", requests=1, context=500, ragged=False, portion=8192,
             model="llama-8b", layers=4, vocab=32000, dtype="float32"),
        # latent attention and routed experts, a few users
        dict(name="kavuvik decode 8", kind="decode", requests=8, context=2000, ragged=True, **kavuvik, **bf16),
        dict(name="kavuvik prefill 3000", kind="prefill", requests=1, context=3000, ragged=False, portion=8192, **kavuvik, **bf16),
        # a recurrence with a state per request, many users
        dict(name="vepitar decode 48", kind="decode", requests=48, context=1000, ragged=True, **vepitar, **bf16),
        # several new prompts in one step
        dict(name="vepitar prefill 4x900", kind="prefill", requests=4, context=900, ragged=True, portion=8192, **vepitar, **bf16),
        # the sampler of a step of a busy server
        dict(name="sample 64", kind="sample", requests=64, vocab=128256, temperature=0.8, top_p=0.9),
    ]


def _log_int(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def draw(rng):
    kind = rng.choice(["decode", "decode", "decode", "prefill", "prefill", "prefill", "serve", "score", "sample"])
    if kind == "sample":
        return dict(kind=kind, requests=_log_int(rng, 1, 64), vocab=rng.choice([32000, 50257, 128256]),
                    temperature=rng.choice([0.6, 0.8, 1.0]), top_p=rng.choice([0.8, 0.9, 0.95]))
    family = rng.choice(["llama", "kavuvik", "vepitar"] if kind in ("decode", "prefill") else ["llama"])
    model = "llama-3b" if kind == "serve" else rng.choice(sorted({"llama": LLAMA, "kavuvik": KAVUVIK, "vepitar": VEPITAR}[family]))
    case = dict(kind=kind, model=model, dtype="float32" if kind == "score" else "bfloat16", ragged=rng.random() < 0.5,
                vocab=rng.choice([32000, 128256]) if family == "llama" and kind != "score" else 32000)
    if family == "llama":
        case["layers"] = rng.randint(2, 4) if kind == "score" else rng.randint(2, 8)
    else:
        case["layers"] = rng.choice([2, 3, 4])
    if kind == "decode":
        case["requests"] = _log_int(rng, 1, 64)
        case["context"] = _log_int(rng, 64, min(8192, 65536 // case["requests"]))
    elif kind == "prefill":
        case["requests"] = rng.choice([1, 1, 2, 3, 6])
        case["context"] = _log_int(rng, 16, 8192 // case["requests"])
        case["portion"] = rng.choice([8192, 8192, 512])
    elif kind == "score":
        case["requests"] = rng.choice([1, 2])
        case["context"] = _log_int(rng, 16, 500 // case["requests"])
        case["portion"] = 8192
    else:
        case.update(requests=rng.randint(2, 16), context=_log_int(rng, 64, 2000), portion=rng.choice([512, 8192]), new=rng.randint(8, 48))
    return case


# -- configurations and weights -------------------------------------------------------------


def _family(case):
    return case["model"].split("-")[0]


def _shape(case):
    return {"llama": LLAMA, "kavuvik": KAVUVIK, "vepitar": VEPITAR}[_family(case)][case["model"]]


def _lengths(case):
    """How many tokens each request has: all alike, or from a quarter of ``context`` up to all of it."""
    n, longest = case["requests"], case["context"]
    if not case["ragged"] or n == 1:
        return [longest] * n
    low = max(1, longest // 4)
    lengths = [low + (longest - low) * i // (n - 1) for i in range(n)]
    random.Random(n * 100003 + longest).shuffle(lengths)
    return lengths


def _config(case):
    s, n = _shape(case), case["layers"]
    if _family(case) == "llama":
        return dict(architectures=["LlamaForCausalLM"], vocab_size=case["vocab"], hidden_size=s["width"], num_hidden_layers=n,
                    num_attention_heads=s["heads"], num_key_value_heads=s["kv_heads"], head_dim=s["dim"],
                    intermediate_size=s["ff"], rms_norm_eps=1e-5, rope_theta=500000.0, max_position_embeddings=131072,
                    rope_scaling=dict(rope_type="llama3", factor=s["factor"], low_freq_factor=1.0, high_freq_factor=4.0,
                                      original_max_position_embeddings=8192), tie_word_embeddings=False)
    if _family(case) == "kavuvik":
        mixer = dict(heads=s["heads"], dim=s["dim"], rot_dim=s["rot_dim"], vdim=s["vdim"], q_rank=s["q_rank"], kv_rank=s["kv_rank"],
                     scale=(s["dim"] + s["rot_dim"]) ** -0.5, rot=dict(base=500000.0, dims=s["rot_dim"]))
        mlp = dict(kind="moe", router=dict(experts=s["experts"], top=s["top"]), expert=dict(ff=s["ff"], limit=KAVUVIK_LIMIT),
                   shared=dict(ff=s["shared_ff"], limit=KAVUVIK_LIMIT))
        return dict(architecture="Kavuvik", vocab=case["vocab"], width=s["width"], embedding=dict(scale=1.0), norm=dict(eps=1e-6),
                    logit_scale=1.0, max_positions=131072,
                    layers=[dict(type="latent_attention", mixer=mixer, mlp=mlp) for _ in range(n)])
    delta = dict(heads=s["delta_heads"], dim=s["delta_dim"], decay_rank=s["decay_rank"])
    attention = dict(heads=s["heads"], kv_heads=s["kv_heads"], dim=s["dim"], vdim=s["dim"], scale=s["dim"] ** -0.5,
                     conv=s["conv"], mask=dict(size=s["window"]))
    moe = dict(kind="moe", router=dict(experts=s["experts"], top=s["top"]), expert=dict(ff=s["expert_ff"]))
    return dict(architecture="Vepitar", vocab=case["vocab"], width=s["width"], norm=dict(eps=1e-6), streams=s["streams"],
                residual_mult=RESIDUAL_MULT, max_positions=131072,
                layers=[dict(type="attention" if i % 4 == 1 else "general_delta", mixer=attention if i % 4 == 1 else delta,
                             mlp=dict(kind="dense", ff=s["dense_ff"]) if i == 0 else moe) for i in range(n)])


def _weights(case, seed):
    """The model's tensors by their names in a model folder, on the GPU, in the element type that
    is served: matrices N(0, 0.02), those that write into the stream smaller with the model's depth."""
    s, n, d, vocab = _shape(case), case["layers"], _shape(case)["width"], case["vocab"]
    dtype = getattr(torch, case["dtype"])
    gen = torch.Generator(device=DEVICE)
    gen.manual_seed(seed)
    out = {}

    def normal(*shape, std=0.02, mean=0.0):
        t = torch.randn(shape, generator=gen, device=DEVICE, dtype=torch.float32)
        return t.mul_(std).add_(mean).to(dtype)

    back = 0.02 / math.sqrt(2 * n)
    embed = torch.randn((vocab, d), generator=gen, device=DEVICE, dtype=torch.float32)

    def router(experts, top, scale=0.5):
        """Directions of the experts; every token's embedding reaches along ``top`` of them."""
        rows = torch.nn.functional.normalize(torch.randn((experts, d), generator=gen, device=DEVICE), dim=1)
        favoured = torch.rand((vocab, experts), generator=gen, device=DEVICE).topk(top, dim=1).indices
        for j in range(top):
            embed.add_(rows[favoured[:, j]], alpha=ROUTING_STRENGTH)
        return (rows * scale).to(dtype)

    if _family(case) == "llama":
        q, kv, ff = s["heads"] * s["dim"], s["kv_heads"] * s["dim"], s["ff"]
        for i in range(n):
            p = f"model.layers.{i}."
            out[p + "input_layernorm.weight"] = normal(d, std=0.05, mean=1.0)
            out[p + "self_attn.q_proj.weight"] = normal(q, d)
            out[p + "self_attn.k_proj.weight"] = normal(kv, d)
            out[p + "self_attn.v_proj.weight"] = normal(kv, d)
            out[p + "self_attn.o_proj.weight"] = normal(d, q, std=back)
            out[p + "post_attention_layernorm.weight"] = normal(d, std=0.05, mean=1.0)
            out[p + "mlp.gate_proj.weight"] = normal(ff, d)
            out[p + "mlp.up_proj.weight"] = normal(ff, d)
            out[p + "mlp.down_proj.weight"] = normal(d, ff, std=back)
        out["model.norm.weight"] = normal(d, std=0.05, mean=1.0)
        # every token has a likely successor, as in a trained model
        successor = torch.randperm(vocab, generator=gen, device=DEVICE)
        head = torch.randn((vocab, d), generator=gen, device=DEVICE, dtype=torch.float32)
        head[successor] += 0.3 * embed
        out["lm_head.weight"] = head.mul_(0.02).to(dtype)
        out["model.embed_tokens.weight"] = embed.to(dtype)
    elif _family(case) == "kavuvik":
        heads, kr = s["heads"], s["kv_rank"]
        for i in range(n):
            p = f"l{i}."
            out[p + "norm1"], out[p + "norm2"] = normal(d, std=0.05, mean=1.0), normal(d, std=0.05, mean=1.0)
            out[p + "mix.dq"] = normal(s["q_rank"], d)
            out[p + "mix.dq.norm"] = normal(s["q_rank"], std=0.05, mean=1.0)
            out[p + "mix.uq"] = normal(heads * (s["dim"] + s["rot_dim"]), s["q_rank"])
            out[p + "mix.dkv"] = normal(kr + s["rot_dim"], d)
            out[p + "mix.dkv.norm"] = normal(kr, std=0.05, mean=1.0)
            out[p + "mix.uk"], out[p + "mix.uv"] = normal(heads * s["dim"], kr, std=0.07), normal(heads * s["vdim"], kr, std=0.07)
            out[p + "mix.g"] = normal(heads * s["vdim"], d)
            out[p + "mix.o"] = normal(d, heads * s["vdim"], std=back)
            out[p + "mlp.router"] = router(s["experts"], s["top"])
            for name, ff in [(f"e{e}", s["ff"]) for e in range(s["experts"])] + [("shared", s["shared_ff"])]:
                out[f"{p}mlp.{name}.gate"], out[f"{p}mlp.{name}.up"] = normal(ff, d), normal(ff, d)
                out[f"{p}mlp.{name}.down"] = normal(d, ff, std=back)
        out["final.norm"], out["head"], out["embed"] = normal(d, std=0.05, mean=1.0), normal(vocab, d), embed.to(dtype)
    else:
        inner, copies = s["delta_heads"] * s["delta_dim"], s["streams"]
        for i in range(n):
            p = f"l{i}."
            out[p + "norm1"], out[p + "norm2"] = normal(d, std=0.05), normal(d, std=0.05)
            for hc in ("hc1", "hc2"):
                out[f"{p}{hc}.in"], out[f"{p}{hc}.out"] = normal(copies, std=0.1, mean=0.6), normal(copies, std=0.1, mean=1.0)
                out[f"{p}{hc}.mix"] = (torch.eye(copies, device=DEVICE) + 0.05 * torch.randn((copies, copies), generator=gen, device=DEVICE)).to(dtype)
            if i % 4 == 1:
                for name, heads in (("q", s["heads"]), ("k", s["kv_heads"]), ("v", s["kv_heads"])):
                    out[f"{p}mix.{name}"] = normal(heads * s["dim"], d)
                    out[f"{p}mix.{name}.conv"] = normal(heads * s["dim"], s["conv"], std=0.5)
                out[p + "mix.pb"] = normal(s["heads"], std=0.5, mean=-4.0)
                out[p + "mix.g"], out[p + "mix.o"] = normal(s["heads"], d), normal(d, s["heads"] * s["dim"], std=back)
            else:
                for name in ("r", "k", "v", "g", "a"):
                    out[f"{p}mix.{name}"] = normal(inner, d)
                out[p + "mix.a.b"], out[p + "mix.w0"] = normal(inner, std=0.7), normal(inner, std=0.7)
                out[p + "mix.w1"], out[p + "mix.w2"] = normal(s["decay_rank"], d), normal(inner, s["decay_rank"], std=0.1)
                out[p + "mix.norm"], out[p + "mix.o"] = normal(inner, std=0.05, mean=1.0), normal(d, inner, std=back)
            if i == 0:
                out[p + "mlp.gate"], out[p + "mlp.up"] = normal(s["dense_ff"], d), normal(s["dense_ff"], d)
                out[p + "mlp.down"] = normal(d, s["dense_ff"], std=back)
            else:
                out[p + "mlp.router"] = router(s["experts"], s["top"])
                for e in range(s["experts"]):
                    out[f"{p}mlp.e{e}.up"], out[f"{p}mlp.e{e}.down"] = normal(s["expert_ff"], d), normal(d, s["expert_ff"], std=back)
        # the table is the head's too: the last norm brings the logits to an ordinary size
        out["final.norm"], out["embed"] = normal(d, std=0.001, mean=-0.98), embed.to(dtype)
    return out


def _token_ids(case, seed, extra):
    """Per request its prompt's ids, and ``extra`` further ids each."""
    rng = np.random.default_rng(seed)
    return [(rng.integers(0, case["vocab"], n, dtype=np.int32), rng.integers(0, case["vocab"], extra, dtype=np.int32))
            for n in _lengths(case)]


DECODE_IDS = 4096  # ids that decoding requests are fed with in turn


# -- what a program holds, and a pass -----------------------------------------------------------


def _runner(case, seed, room, graphs):
    """``room``: tokens of cache per request beyond its prompt."""
    _, config = parse_config(_config(case))
    lengths = _lengths(case)
    pool = sum(-(-(n + room) // PAGE) * PAGE for n in lengths) + PAGE * len(lengths)
    runner = ModelRunner.from_random(
        config, seed=0,
        server_config=ServerConfig(
            kv_cache_num_tokens=pool, max_seqs_per_forward=len(lengths), max_tokens_per_forward=LONGEST_STEP,
            max_prefill_tokens=LONGEST_STEP, chunked_prefill_size=case.get("portion", LONGEST_STEP), page_size=PAGE,
            use_cudagraph=graphs, cudagraph_max_batch_size=len(lengths), cudagraph_step=1, scheduling_steps_ahead=1),
        model_config=ModelConfig(dtype=case["dtype"], context_len=max(lengths) + room))
    runner.load_state_dict(_weights(case, seed))
    return runner


def _feed(runner, slots, prompts, portion, want):
    """The prompts in steps of at most ``portion`` tokens each and ``LONGEST_STEP`` together; the
    logits that ``want`` asks for (a prompt's length -> wanted places), in the prompts' order."""
    at, logits = [0] * len(slots), []
    while True:
        segments, left = [], LONGEST_STEP
        for i, (slot, ids) in enumerate(zip(slots, prompts)):
            n = min(len(ids) - at[i], portion, left)
            if n > 0:
                places = [w - at[i] for w in want(len(ids)) if at[i] <= w < at[i] + n]
                segments.append(Segment(slot, at[i], ids[at[i]: at[i] + n], places))
                at[i] += n
                left -= n
        if not segments:
            return logits
        got = runner.step(segments)
        row = 0
        for seg in segments:
            if seg.want:
                logits.append((seg.slot, seg.start, got[row: row + len(seg.want)]))
                row += len(seg.want)


def _begin(state):
    """New requests whose prompts are in the cache."""
    runner, prompts = state["runner"], [ids for ids, _ in state["ids"]]
    state["slots"] = [runner.admit() for _ in prompts]
    _feed(runner, state["slots"], prompts, LONGEST_STEP, lambda n: [])
    state["step"] = 0


def _room(case):
    return 4096 if case["requests"] > 8 else 12288


def prepare(case, seed):
    case = dict(case)
    if case["kind"] == "sample":
        gen = torch.Generator(device=DEVICE)
        gen.manual_seed(seed)
        n = case["requests"]
        # the logits of a language model: a broad base and a few likely tokens
        logits = torch.randn((n, case["vocab"]), generator=gen, device=DEVICE) * 2.0
        likely = torch.randint(0, case["vocab"], (n, 32), generator=gen, device=DEVICE)
        logits.scatter_add_(1, likely, 12.0 * torch.rand((n, 32), generator=gen, device=DEVICE))
        params = [SamplingParams(temperature=case["temperature"], top_p=case["top_p"]) for _ in range(n)]
        seeds = [int(v) for v in np.random.default_rng(seed).integers(0, 1 << 62, n)]
        return dict(case=case, sampler=Sampler(DEVICE), logits=logits, params=params, seeds=seeds, draws=list(range(n)))
    if case["kind"] == "decode":
        state = dict(case=case, runner=_runner(case, seed, _room(case), graphs=True), ids=_token_ids(case, seed, DECODE_IDS))
        state["runner"].capture_graphs([case["requests"]])
        _begin(state)
        return state
    if case["kind"] == "serve":
        engine = InferenceEngine(_runner(case, seed, case["new"] + PAGE, graphs=True), None, seed=0)
        engine.initialize(capture_graphs=True)
        params = SamplingParams(max_new_tokens=case["new"], temperature=0.0, ignore_eos=True)
        return dict(case=case, engine=engine, requests=[(ids.tolist(), params) for ids, _ in _token_ids(case, seed, 0)])
    return dict(case=case, runner=_runner(case, seed, PAGE, graphs=False), ids=_token_ids(case, seed, 0))


def run(state):
    case, kind = state["case"], state["case"]["kind"]
    if kind == "sample":
        tokens, logprobs = state["sampler"].forward(state["logits"], state["params"], state["seeds"], state["draws"])
        return {"tokens": tokens, "logprobs": logprobs}
    if kind == "serve":
        results = state["engine"].infer_batch(state["requests"])
        return {"tokens": np.array([r.output_ids[0] for r in results], dtype=np.int64),
                "logprobs": np.array([r.output_logprobs[0] for r in results], dtype=np.float32)}
    runner = state["runner"]
    if kind == "decode":
        if state["step"] >= _room(case):  # the requests have come to their end: the next ones
            for slot in state["slots"]:
                runner.free(slot)
            _begin(state)
        k = state["step"] % DECODE_IDS
        state["step"] += 1
        return {"logits": runner.step([Segment(slot, runner.cache.length(slot), ids[k: k + 1], [0])
                                       for slot, (_, ids) in zip(state["slots"], state["ids"])])}
    prompts = [ids for ids, _ in state["ids"]]
    slots = [runner.admit() for _ in prompts]
    want = (lambda n: list(range(n))) if kind == "score" else (lambda n: [n - 1])
    got = _feed(runner, slots, prompts, case["portion"], want)
    for slot in slots:
        runner.free(slot)
    if len(got) == 1:
        return {"logits": got[0][2]}
    got.sort(key=lambda entry: (slots.index(entry[0]), entry[1]))
    return {"logits": torch.cat([rows for _, _, rows in got])}


# -- what a pass cannot do without ----------------------------------------------------------------


def _counts(case, rows):
    """Per model: the weights that every token meets (entries), those of which ``rows`` tokens reach
    a part (entries read), floating operations a token for the linear layers, and per layer kind
    what attention and recurrences take."""
    s, n, d = _shape(case), case["layers"], _shape(case)["width"]
    if _family(case) == "llama":
        q, kv = s["heads"] * s["dim"], s["kv_heads"] * s["dim"]
        dense = n * (d * (q + 2 * kv) + q * d + 3 * d * s["ff"])
        return dict(dense=dense, routed=0, reached=0, key_bytes=n * 2 * kv, pair_flops=4.0 * n * q, window=0, state=0, state_flops=0.0)
    reach = lambda experts, top: experts * (1.0 - (1.0 - top / experts) ** rows)  # noqa: E731
    if _family(case) == "kavuvik":
        h = s["heads"]
        dense = d * (s["q_rank"] + s["kv_rank"] + s["rot_dim"] + h * s["vdim"] + s["experts"]) + s["q_rank"] * h * (s["dim"] + s["rot_dim"])
        dense += h * s["vdim"] * d + h * (s["dim"] + s["vdim"]) * s["kv_rank"] + 3 * d * s["shared_ff"]
        expert = 3 * d * s["ff"]
        cached = s["kv_rank"] + s["rot_dim"]
        return dict(dense=n * dense, routed=n * s["top"] * expert, reached=n * reach(s["experts"], s["top"]) * expert,
                    key_bytes=n * cached, pair_flops=2.0 * n * h * (s["dim"] + s["rot_dim"] + s["vdim"]), window=0, state=0, state_flops=0.0)
    n_att = sum(i % 4 == 1 for i in range(n))
    n_delta, n_moe = n - n_att, n - 1
    q, kv, inner = s["heads"] * s["dim"], s["kv_heads"] * s["dim"], s["delta_heads"] * s["delta_dim"]
    dense = n_att * (d * (q + 2 * kv + s["heads"]) + q * d) + n_delta * (6 * d * inner + (d + inner) * s["decay_rank"])
    dense += 3 * d * s["dense_ff"] + n_moe * d * s["experts"]
    expert = 2 * d * s["expert_ff"]
    state = n_delta * inner * s["delta_dim"]
    return dict(dense=dense, routed=n_moe * s["top"] * expert, reached=n_moe * reach(s["experts"], s["top"]) * expert,
                key_bytes=n_att * 2 * kv, pair_flops=4.0 * n_att * q, window=s["window"], state=state, state_flops=9.0 * state)


def _pairs(n, window):
    """(query, key) pairs of a prompt of ``n`` tokens that sees itself causally."""
    if window and n > window:
        return window * (window + 1) / 2 + (n - window) * window
    return n * (n + 1) / 2


def work(case):
    if case["kind"] == "sample":
        n = case["requests"] * case["vocab"]
        return {"bytes": 4.0 * n + 8.0 * case["requests"], "flops": 4.0 * n}
    elt = 2 if case["dtype"] == "bfloat16" else 4
    lengths, d, vocab = _lengths(case), _shape(case)["width"], case["vocab"]
    if case["kind"] == "decode":
        rows = len(lengths)
        c = _counts(case, rows)
        keys = sum(min(n + 1, c["window"]) if c["window"] else n + 1 for n in lengths)
        by = elt * (c["dense"] + c["reached"] + vocab * d + rows * d + keys * c["key_bytes"]) + rows * (8.0 * c["state"] + 4.0 * vocab)
        fl = rows * (2.0 * (c["dense"] + c["routed"] + vocab * d) + c["state_flops"]) + keys * c["pair_flops"]
        return {"bytes": by, "flops": fl}
    tokens = sum(lengths)
    wanted = tokens if case["kind"] == "score" else len(lengths)
    c = _counts(case, tokens)
    by = elt * (c["dense"] + c["reached"] + vocab * d + tokens * (d + c["key_bytes"])) + 4.0 * wanted * vocab + 4.0 * len(lengths) * c["state"]
    fl = tokens * (2.0 * (c["dense"] + c["routed"]) + c["state_flops"]) + 2.0 * wanted * vocab * d
    fl += sum(_pairs(n, c["window"]) for n in lengths) * c["pair_flops"]
    if case["kind"] == "serve":  # and then the steps that decode all requests but their first token
        steps, rows = case["new"] - 1, len(lengths)
        c = _counts(case, rows)
        keys = sum(n + (case["new"] + 1) / 2.0 for n in lengths)
        by += steps * (elt * (c["dense"] + vocab * d + rows * d + keys * c["key_bytes"]) + rows * 8.0)
        fl += steps * (rows * 2.0 * (c["dense"] + vocab * d) + keys * c["pair_flops"])
    return {"bytes": by, "flops": fl}


def tolerance(case):
    """About four times the largest distance from ``exact`` that this engine showed over the listed
    cases and 40 drawn ones (logits of Llama layers 0.0088, of Kavuvik's 0.003, of Vepitar's 0.002,
    whose embeddings weigh most in the stream; float32 1.5e-6; served log-probabilities 0.0036)."""
    if case["kind"] == "sample":
        return {"rel": 1.5e-6, "max": 1e-5, "differ": 0.0}
    if case["dtype"] == "float32":
        return {"rel": 6e-6, "max": 4e-5}
    if case["kind"] == "serve":
        return {"rel": 0.015, "max": 0.05, "differ": 0.0}
    rel, largest = {"llama": (0.03, 0.16), "kavuvik": (0.012, 0.06), "vepitar": (0.008, 0.04)}[_family(case)]
    return {"rel": rel, "max": largest}


# -- the same in 64 bits ----------------------------------------------------------------------------


def _product(x, w):
    """``x @ w.T`` in 64 bits, in stretches of rows that keep what lies in between small."""
    w = w.to(F64)
    return torch.cat([part @ w.T for part in x.split(8192)])


def _unit(x, eps):
    return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + eps)


def _frequencies(base, dims, scaling=None):
    """Rotation frequencies, in the float32 that the designs state them in; ``scaling``: the
    stretching of long wavelengths by bands."""
    freq = 1.0 / (base ** (torch.arange(0, dims, 2, dtype=torch.float32) / dims))
    if scaling:
        out = []
        for f in freq:
            wave = 2 * math.pi / f
            if wave < scaling["original_max_position_embeddings"] / scaling["high_freq_factor"]:
                out.append(f)
            elif wave > scaling["original_max_position_embeddings"] / scaling["low_freq_factor"]:
                out.append(f / scaling["factor"])
            else:
                r = (scaling["original_max_position_embeddings"] / wave - scaling["low_freq_factor"]) / (
                    scaling["high_freq_factor"] - scaling["low_freq_factor"])
                out.append((1 - r) * f / scaling["factor"] + r * f)
        freq = torch.stack(out).to(torch.float32)
    return freq.to(DEVICE)


def _rotate(x, freq, first=0):
    """``x`` [T, heads, D]: entry i of the first 2 * len(freq) turns with entry i + len(freq);
    the tokens stand at the positions from ``first`` on."""
    positions = torch.arange(first, first + x.shape[0], device=DEVICE, dtype=torch.float32)
    angle = (positions[:, None] * freq[None, :]).to(F64)[:, None, :]
    cos, sin, half = torch.cos(angle), torch.sin(angle), freq.numel()
    u, v = x[..., :half], x[..., half: 2 * half]
    return torch.cat((u * cos - v * sin, v * cos + u * sin, x[..., 2 * half:]), -1)


def _heads_attention(q, k, v, scale, window=0, bias=None, last=None):
    """``q`` [Q, H, D] of the last Q tokens against ``k``, ``v`` [T, G, D] of all of them, causal: softmax, or
    sigmoid with ``bias`` [H]."""
    Q, H, _ = q.shape
    T, G = k.shape[0], k.shape[1]
    out = torch.empty((Q, H, v.shape[2]), dtype=F64, device=q.device)
    place = torch.arange(T, device=q.device)
    step = max(1, min(Q, (1 << 27) // T))
    for a in range(0, Q, step):
        b = min(Q, a + step)
        gap = (T - Q + torch.arange(a, b, device=q.device))[:, None] - place[None, :]
        hidden = (gap < 0) | (gap >= window) if window else gap < 0
        for h in range(H):
            g = h // (H // G)
            s = (q[a:b, h] @ k[:, g].T.contiguous()) * scale
            if bias is None:
                w = torch.softmax(s.masked_fill(hidden, -math.inf), -1)
            else:
                w = torch.sigmoid(s + bias[h]).masked_fill(hidden, 0.0)
            out[a:b, h] = w @ v[:, g].contiguous()
    return out


def _by_request(lengths, fn, *arrays):
    """``fn`` on every request's rows of the arrays."""
    return torch.cat([fn(*part) for part in zip(*(a.split(lengths) for a in arrays))])


def _route(logits, top, weigh):
    """Chosen experts, and their scores over the chosen ones' sum."""
    scores, chosen = torch.topk(weigh(logits), top, dim=-1)
    return chosen, scores / (scores.sum(-1, keepdim=True) + 1e-20)


def _experts(h, chosen, weight, n_experts, expert):
    out = torch.zeros_like(h)
    for e in range(n_experts):
        rows, place = (chosen == e).nonzero(as_tuple=True)
        if rows.numel():
            out.index_add_(0, rows, expert(e, h[rows]) * weight[rows, place][:, None])
    return out


def _llama_stream(case, w, ids, lengths, cache=None):
    """The stream after the last layer for the tokens ``ids`` (``lengths`` of them a request).
    ``cache``: a list of (keys, values) per request and layer that is read and extended."""
    s, cfg = _shape(case), _config(case)
    freq = _frequencies(cfg["rope_theta"], s["dim"], cfg["rope_scaling"])
    eps = cfg["rms_norm_eps"]
    x = w["model.embed_tokens.weight"][ids].to(F64)
    for i in range(case["layers"]):
        p = f"model.layers.{i}."
        h = _unit(x, eps) * w[p + "input_layernorm.weight"].to(F64)
        q, k, v = (_product(h, w[f"{p}self_attn.{name}_proj.weight"]).view(len(ids), -1, s["dim"]) for name in "qkv")
        parts = []
        for r, (qr, kr, vr) in enumerate(zip(q.split(lengths), k.split(lengths), v.split(lengths))):
            before = cache[r][i] if cache is not None and cache[r][i] is not None else None
            first = 0 if before is None else before[0].shape[0]
            qr, kr = _rotate(qr, freq, first), _rotate(kr, freq, first)
            if before is not None:
                kr, vr = torch.cat((before[0], kr)), torch.cat((before[1], vr))
            if cache is not None:
                cache[r][i] = (kr, vr)
            parts.append(_heads_attention(qr, kr, vr, s["dim"] ** -0.5))
        del q, k, v
        x = x + _product(torch.cat(parts).reshape(len(ids), -1), w[p + "self_attn.o_proj.weight"])
        h = _unit(x, eps) * w[p + "post_attention_layernorm.weight"].to(F64)
        for rows in torch.arange(len(ids), device=DEVICE).split(8192):
            g = _product(h[rows], w[p + "mlp.gate_proj.weight"])
            x[rows] += _product(g * torch.sigmoid(g) * _product(h[rows], w[p + "mlp.up_proj.weight"]), w[p + "mlp.down_proj.weight"])
    return x


def _llama_logits(w, x):
    return _product(_unit(x, 1e-5) * w["model.norm.weight"].to(F64), w["lm_head.weight"])


def _kavuvik_stream(case, w, ids, lengths):
    s, eps = _shape(case), 1e-6
    freq = _frequencies(500000.0, s["rot_dim"])
    h_, dn, kr = s["heads"], s["dim"], s["kv_rank"]
    x = w["embed"][ids].to(F64)

    def gated(g, u):
        g, u = g.clamp(max=KAVUVIK_LIMIT), u.clamp(-KAVUVIK_LIMIT, KAVUVIK_LIMIT)
        return g * torch.sigmoid(KAVUVIK_ALPHA * g) * (u + 1)

    for i in range(case["layers"]):
        p = f"l{i}."
        t = lambda name, p=p: w[p + name].to(F64)  # noqa: E731
        h = _unit(x, eps) * t("norm1")
        q = _product(_unit(_product(h, t("mix.dq")), eps) * t("mix.dq.norm"), t("mix.uq")).view(len(ids), h_, -1)
        down = _product(h, t("mix.dkv"))
        c = _unit(down[:, :kr], eps) * t("mix.dkv.norm")
        keys, values = _product(c, t("mix.uk")).view(len(ids), h_, dn), _product(c, t("mix.uv")).view(len(ids), h_, -1)

        def attend(qr, turning, k, v):
            qr = torch.cat((qr[..., :dn], _rotate(qr[..., dn:], freq)), -1)
            turned = _rotate(turning[:, None, :], freq).expand(-1, h_, -1)
            return _heads_attention(qr, torch.cat((k, turned), -1), v, (dn + s["rot_dim"]) ** -0.5)

        out = _by_request(lengths, attend, q, down[:, kr:], keys, values).reshape(len(ids), -1) * torch.sigmoid(_product(h, t("mix.g")))
        delta = _product(out, t("mix.o"))
        h = _unit(x, eps) * t("norm2")
        chosen, weight = _route(_product(h, t("mlp.router")), s["top"], torch.sigmoid)
        ff = lambda name, rows: _product(gated(_product(rows, t(f"mlp.{name}.gate")), _product(rows, t(f"mlp.{name}.up"))),  # noqa: E731
                                         t(f"mlp.{name}.down"))
        x = x + delta + ff("shared", h) + _experts(h, chosen, weight, s["experts"], lambda e, rows: ff(f"e{e}", rows))
    return x


def _kavuvik_logits(w, x):
    return _product(_unit(x, 1e-6) * w["final.norm"].to(F64), w["head"])


def _convolve(u, taps):
    """Causal convolution over time of every channel; the last tap is the token's own."""
    n = taps.shape[1]
    padded = torch.cat((u.new_zeros((n - 1, u.shape[1])), u))
    return sum(taps[:, j] * padded[j: j + u.shape[0]] for j in range(n))


def _delta_reads(lengths, r, k, v, decay, a):
    """The generalized delta rule over all requests side by side ([T, H, D] each, request after
    request): the old state is decayed, loses what it holds along the unit key, gains the
    key's value, and is read."""
    longest = max(lengths)
    pad = lambda t: torch.stack([torch.cat((part, part.new_zeros((longest - len(part), *part.shape[1:])))) for part in t.split(lengths)], 1)  # noqa: E731
    r, k, v, decay, a = (pad(t) for t in (r, k, v, decay, a))  # [longest, requests, H, D]
    unit = k * torch.rsqrt((k * k).sum(-1, keepdim=True) + 1e-6)
    S = torch.zeros((*k.shape[1:], k.shape[-1]), dtype=F64, device=k.device)
    out = torch.empty_like(v)
    for t in range(longest):
        held = (unit[t][..., None] * S).sum(-2)
        S = decay[t][..., None] * S - (a[t] * unit[t])[..., None] * held[..., None, :] + k[t][..., None] * v[t][..., None, :]
        out[t] = (r[t][..., None] * S).sum(-2)
    return torch.cat([out[:n, i] for i, n in enumerate(lengths)])


def _vepitar_stream(case, w, ids, lengths):
    s, eps, n = _shape(case), 1e-6, len(ids)
    streams = [w["embed"][ids].to(F64) for _ in range(s["streams"])]
    for i in range(case["layers"]):
        p = f"l{i}."
        t = lambda name, p=p: w[p + name].to(F64)  # noqa: E731
        for part in (1, 2):
            inp = sum(t(f"hc{part}.in")[c] * x for c, x in enumerate(streams))
            h = _unit(inp, eps) * (1.0 + t(f"norm{part}"))
            if part == 1 and i % 4 == 1:
                q, k, v = (_unit(_by_request(lengths, lambda u: _convolve(u, t(f"mix.{name}.conv")), _product(h, t(f"mix.{name}")))
                                 .view(n, -1, s["dim"]), eps) for name in "qkv")
                out = _by_request(lengths, lambda q, k, v: _heads_attention(q, k, v, s["dim"] ** -0.5, s["window"], t("mix.pb")), q, k, v)
                y = _product((out * torch.sigmoid(_product(h, t("mix.g")))[..., None]).reshape(n, -1), t("mix.o"))
            elif part == 1:
                heads = lambda u: u.view(n, s["delta_heads"], s["delta_dim"])  # noqa: E731
                z = _product(torch.tanh(_product(h, t("mix.w1"))), t("mix.w2")) + t("mix.w0")
                decay = torch.exp(-math.exp(-0.5) * torch.sigmoid(z))
                a = torch.sigmoid(_product(h, t("mix.a")) + t("mix.a.b"))
                reads = _delta_reads(lengths, *(heads(_product(h, t(f"mix.{name}"))) for name in "rkv"), heads(decay), heads(a))
                y = _unit(reads, eps).reshape(n, -1) * t("mix.norm") * torch.sigmoid(_product(h, t("mix.g")))
                y = _product(y, t("mix.o"))
            elif i == 0:
                g = _product(h, t("mlp.gate"))
                y = _product(g * torch.sigmoid(g) * _product(h, t("mlp.up")), t("mlp.down"))
            else:
                chosen, weight = _route(_product(h, t("mlp.router")), s["top"], lambda z: torch.softmax(z, -1))
                y = _experts(h, chosen, weight, s["experts"], lambda e, rows: _product(
                    torch.relu(_product(rows, t(f"mlp.e{e}.up"))) ** 2, t(f"mlp.e{e}.down")))
            mix, to = t(f"hc{part}.mix"), t(f"hc{part}.out")
            streams = [sum(mix[b, c] * streams[b] for b in range(len(streams))) + RESIDUAL_MULT * to[c] * y for c in range(len(streams))]
    return sum(streams)


def _vepitar_logits(w, x):
    return _product(_unit(x, 1e-6) * (1.0 + w["final.norm"].to(F64)), w["embed"])


def _exact_sample(case, seed):
    state = prepare(case, seed)
    z = state["logits"].to(F64) / case["temperature"]
    logp = torch.log_softmax(z, -1)
    p, order = torch.exp(logp).sort(-1, descending=True)
    before = p.cumsum(-1) - p
    kept = torch.zeros_like(p).scatter_(1, order, torch.where(before <= case["top_p"], p, 0.0))
    mask = (1 << 64) - 1
    u = []
    for s, index in zip(state["seeds"], state["draws"]):  # the request's counter-based generator
        x = (s * 0x9E3779B97F4A7C15 + (index + 1) * 0xD1B54A32D192ED03) & mask
        x = ((x ^ (x >> 30)) * 0xBF58476D1CE4E5B9) & mask
        x = ((x ^ (x >> 27)) * 0x94D049BB133111EB) & mask
        u.append(((x ^ (x >> 31)) >> 40) / 16777216.0)
    along = kept.cumsum(-1)
    tokens = (along > torch.tensor(u, dtype=F64, device=DEVICE)[:, None] * along[:, -1:]).to(torch.int8).argmax(-1)
    return {"tokens": None, "logprobs": logp.gather(1, tokens[:, None])[:, 0]}


@torch.no_grad()
def exact(case, seed):
    if case["kind"] == "sample":
        return _exact_sample(case, seed)
    lengths = _lengths(case)
    tokens = sum(lengths)
    c = _counts(case, tokens)
    if 2.0 * tokens * (c["dense"] + c["routed"]) + 2.0 * sum(n * n for n in lengths) * c["pair_flops"] > EXACT_FLOPS:
        return None
    w = _weights(case, seed)
    ids = _token_ids(case, seed, DECODE_IDS if case["kind"] == "decode" else 0)
    on_gpu = lambda arrays: torch.from_numpy(np.concatenate(arrays)).to(DEVICE, torch.int64)  # noqa: E731
    if case["kind"] == "serve":
        cache = [[None] * case["layers"] for _ in lengths]
        x = _llama_stream(case, w, on_gpu([prompt for prompt, _ in ids]), lengths, cache)
        x = torch.stack([part[-1] for part in x.split(lengths)])
        logprobs = []
        for step in range(case["new"]):
            logp = torch.log_softmax(_llama_logits(w, x), -1)
            best, token = logp.max(-1)
            logprobs.append(best)
            if step + 1 < case["new"]:
                x = _llama_stream(case, w, token, [1] * len(lengths), cache)
        return {"tokens": None, "logprobs": torch.stack(logprobs, 1)}
    stream, logits = {"llama": (_llama_stream, _llama_logits), "kavuvik": (_kavuvik_stream, _kavuvik_logits),
                      "vepitar": (_vepitar_stream, _vepitar_logits)}[_family(case)]
    if case["kind"] == "decode":
        ids = [np.concatenate((prompt, more[:1])) for prompt, more in ids]
    else:
        ids = [prompt for prompt, _ in ids]
    x = stream(case, w, on_gpu(ids), [len(i) for i in ids])
    if case["kind"] != "score":
        x = torch.stack([part[-1] for part in x.split([len(i) for i in ids])])
    return {"logits": logits(w, x)}
