"""What the engine's speed is measured on: steps of whole models, as serving meets them.

A case is a model (a design, its shape, its layer count, its type) and what one stretch of serving brings:

* ``decoding`` requests that each hold ``cached`` tokens already (their pages come from the prefix index, as a
  conversation's next turn finds them) and bring one token to every step;
* ``prompts``: the lengths of further prompts that arrive at once, each behind ``behind`` cached tokens; they run in
  steps of at most ``budget`` tokens beside the decoding requests' single tokens, first come, first served;
* ``steps`` decode steps after that, in which every request brings one token.

A pass admits the requests, runs the steps through the engine's step function, keeps every step's logits and releases
the requests, so that it can be run again.  The tokens are given (scoring and replay do the same), so that two
implementations see the same ones whatever their last bit says.

The models have 12 layers (the 7B shape 8) of their 24 to 36: a layer costs the same however many follow it, and the
16-bit roundings that random weights amplify from layer to layer stay small enough to compare two runs.

Weights are random, N(0, 0.02) and 1 + N(0, 0.02) for norms, token ids uniform, as in the engine's benchmark.
"""

from __future__ import annotations

import math
import zlib

import torch

from cie_amd.config import build_engine_config, config_from_dict
from cie_amd.engine.loading import build_model
from cie_amd.engine.runner import Runner, StepEntry
from cie_amd.workloads import SHAPES

PAGE = 16

# the first tiny configuration that the baseline record names
TINY = dict(model_type="qwen2", hidden_size=64, num_hidden_layers=2, num_attention_heads=4, num_key_value_heads=2,
            intermediate_size=128, vocab_size=256, rope_theta=10000.0, rms_norm_eps=1e-6, attention_bias=True,
            tie_word_embeddings=True, use_sliding_window=False, max_position_embeddings=128)


def _case(name=None, design="qwen2", shape="3b", layers=12, dtype="bfloat16", decoding=0, cached=0, prompts="",
          behind=0, budget=2048, steps=0):
    case = dict(design=design, shape=shape, layers=layers, dtype=dtype, decoding=decoding, cached=cached,
                prompts=prompts, behind=behind, budget=budget, steps=steps)
    return dict(case, name=name) if name else case


def listed():
    return [
        # the smallest model there is, three short prompts and eight tokens each, in 32 bits: launches and latency only
        _case("tiny-fp32", shape="tiny", layers=2, dtype="float32", prompts="5,17,33", budget=64, steps=8),
        # one user's conversation: decode steps of one sequence
        _case("3b-decode-1", decoding=1, cached=2032, steps=16),
        # the benchmark's headline: eight sequences at a context of 4,096
        _case("3b-decode-8", decoding=8, cached=4064, steps=16),
        # a busy server: many sequences, shorter contexts
        _case("3b-decode-64", decoding=64, cached=1008, steps=8),
        # the benchmark's prefill: one prompt that fills the token budget
        _case("3b-prompt-2048", prompts="2048"),
        # short questions that arrive together, and their first answers' tokens
        _case("3b-prompts-ragged", prompts="37,311,129,64,72", steps=2),
        # chunked serving: eight decoding sequences beside a long prompt that comes in portions of 248 tokens
        _case("3b-mixed-256", decoding=8, cached=2000, prompts="744", budget=256),
        # a longer message in a conversation: a prompt that is no round number, behind a cached history
        _case("7b-turn", shape="7b", layers=8, prompts="777", behind=4000, steps=4),
        # the 32-bit path over a prompt: the reference output that a 16-bit run is compared with
        _case("3b-prompt-fp32", dtype="float32", prompts="517"),
        # ... and token by token
        _case("3b-decode-4-fp32", dtype="float32", decoding=4, cached=1008, steps=8),
        # the engine's second design: retention, latent attention and a gated recurrence in turn, over a prompt
        _case("polosun-prompt", design="polosun", prompts="1999"),
        # ... and eight short conversations of it
        _case("polosun-decode-8", design="polosun", prompts="61,128,97,33,80,111,20,49", steps=24),
    ]


def _log(rng, low, high):
    return max(low, min(high, round(math.exp(rng.uniform(math.log(low), math.log(high))))))


def draw(rng):
    kind = rng.choice(("tiny", "decode", "decode", "prompt", "prompts", "mixed", "turn", "prompt-fp32", "decode-fp32",
                       "polosun", "polosun-decode"))
    shape = rng.choice(("0.5b", "3b"))
    layers = 12
    if kind == "tiny":
        lengths = [rng.randint(1, 40) for _ in range(rng.randint(1, 6))]
        return _case(shape="tiny", layers=2, dtype=rng.choice(("float32", "bfloat16")), prompts=",".join(map(str, lengths)),
                     budget=rng.choice((48, 64)), steps=rng.randint(1, 12))
    if kind == "decode":
        requests = _log(rng, 1, 64)
        return _case(shape=shape, layers=layers, decoding=requests, steps=8,
                     cached=PAGE * _log(rng, 4, max(8, min(254, 4032 // requests))))
    if kind == "prompt":
        return _case(shape=shape, layers=layers, prompts=str(_log(rng, 100, 2048)))
    if kind == "prompts":
        lengths = [_log(rng, 16, 500) for _ in range(rng.randint(2, 6))]
        return _case(shape=shape, layers=layers, prompts=",".join(map(str, lengths)), steps=rng.randint(1, 3))
    if kind == "mixed":
        requests, portion = _log(rng, 2, 32), _log(rng, 16, 500)
        return _case(shape=shape, layers=layers, decoding=requests, cached=PAGE * _log(rng, 8, 2000 // requests),
                     prompts=str(2 * portion), budget=requests + portion)
    if kind == "turn":
        return _case(shape=shape, layers=layers, prompts=str(_log(rng, 30, 900)), behind=PAGE * _log(rng, 16, 250),
                     steps=rng.randint(1, 4))
    if kind == "prompt-fp32":
        return _case(shape=shape, layers=layers, dtype="float32", prompts=str(_log(rng, 20, 500)))
    if kind == "decode-fp32":
        requests = _log(rng, 1, 16)
        return _case(shape=shape, layers=layers, dtype="float32", decoding=requests, steps=4,
                     cached=PAGE * _log(rng, 4, 1008 // requests))
    if kind == "polosun":
        return _case(design="polosun", shape=shape, layers=rng.choice((6, 9, 12)), prompts=str(_log(rng, 100, 2000)))
    lengths = [_log(rng, 8, 250) for _ in range(_log(rng, 1, 12))]
    return _case(design="polosun", shape=shape, layers=rng.choice((6, 9, 12)), prompts=",".join(map(str, lengths)),
                 steps=rng.randint(4, 16))


# ---------------------------------------------------------------- the model
def _raw(case):
    if case["shape"] == "tiny":
        return dict(TINY, architectures=["Qwen2ForCausalLM"])
    shape = SHAPES[case["shape"]]
    if case["design"] == "qwen2":
        return dict(shape, architectures=["Qwen2ForCausalLM"], num_hidden_layers=case["layers"])
    # the benchmark's Polosun: heads of 128 x 256 for the retention, a latent of 96 and a turned part of 32 for the
    # attention, a recurrence in blocks of 256 channels with four taps (a narrow model: blocks of 128)
    width = shape["hidden_size"]
    mlp = {"kind": "dense", "ff": shape["intermediate_size"]}
    heads, block = max(1, width // 256), 256 if width % 256 == 0 else 128
    kinds = [
        {"type": "retention", "mlp": mlp,
         "mixer": {"heads": heads, "dim": 128, "vdim": 256, "rot": {"base": 10000.0, "dims": 128},
                   "decay": [1.0 - 2.0 ** (-5 - 3 * h / max(heads - 1, 1)) for h in range(heads)]}},
        {"type": "latent_attention", "mlp": mlp,
         "mixer": {"heads": width // 128, "dim": 128, "rot_dim": 32, "vdim": 128, "kv_rank": 96, "scale": 160 ** -0.5,
                   "rot": {"base": 1000000.0, "dims": 32,
                           "scaling": {"factor": 4.0, "fast": 32.0, "original": 8192, "slow": 1.0}}}},
        {"type": "rglru", "mlp": mlp, "mixer": {"width": width, "blocks": width // block, "conv": 4}},
    ]
    return {"architecture": "Polosun", "vocab": shape["vocab_size"], "width": width, "residual_mult": 0.5,
            "norm": {"eps": 1e-6}, "layers": [kinds[i % 3] for i in range(case["layers"])]}


def _tensor(name, shape, seed, dtype):
    """The model's tensor of this name: N(0, 0.02), norms and the weights of a depth average 1 + N(0, 0.02)."""
    g = torch.Generator(device="cuda")
    g.manual_seed(zlib.crc32(name.encode()) + (int(seed) << 32))
    values = torch.randn(tuple(shape), generator=g, device="cuda") * 0.02
    if "norm" in name or name.endswith("dwa"):
        values += 1.0
    return values.to(getattr(torch, dtype))


class _Weights:
    """A source of a model's tensors, each made when it is asked for."""

    def __init__(self, seed):
        self.seed = seed

    def load(self, expected, dtype, device, tied_optional=None):
        return _Drawn(expected, self.seed, dtype)

    open = load


class _Drawn:
    def __init__(self, expected, seed, dtype):
        self.expected, self.seed, self.dtype = expected, seed, dtype

    def __contains__(self, name):
        return name in self.expected

    def __iter__(self):
        return iter(self.expected)

    def __getitem__(self, name):
        return _tensor(name, self.expected[name].random_shape, self.seed, self.dtype)

    def get(self, name, default=None):
        return self[name] if name in self else default


def _prompts(case):
    return [int(n) for n in case["prompts"].split(",") if n]


def _requests(case):
    """(cached tokens, tokens that the pass brings) of every request: those that decode, then the prompts."""
    phase = len(_prompt_steps(case))
    held = [(case["cached"], phase + case["steps"])] * case["decoding"]
    return held + [(case["behind"], n + case["steps"]) for n in _prompts(case)]


def _prompt_steps(case):
    """The steps that bring prompt tokens: for each the (prompt, first token, count) portions."""
    steps, room, at = [], 0, []
    for index, count in enumerate(_prompts(case)):
        first = 0
        while first < count:
            if room == 0:
                at = []
                steps.append(at)
                room = case["budget"] - case["decoding"]
            take = min(room, count - first)
            at.append((index, first, take))
            first += take
            room -= take
    return steps


def _schedule(case):
    """Every step of a pass: a list of (request, first of its new tokens, count, whether the last one's logits are wanted)."""
    out, lengths, waiting = [], _prompts(case), case["decoding"]
    for number, portions in enumerate(_prompt_steps(case)):
        step = [(r, number, 1, True) for r in range(waiting)]
        step += [(waiting + index, first, take, first + take == lengths[index]) for index, first, take in portions]
        out.append(step)
    phase = len(out)
    for k in range(case["steps"]):
        out.append([(r, phase + k, 1, True) for r in range(waiting)]
                   + [(waiting + index, n + k, 1, True) for index, n in enumerate(lengths)])
    return out


def _tokens(case, seed, vocab):
    """All tokens of every request, the cached ones first."""
    g = torch.Generator().manual_seed(int(seed) * 7919 + 17)
    return [torch.randint(0, vocab, (held + new,), generator=g).tolist() for held, new in _requests(case)]


def prepare(case, seed):
    raw = _raw(case)
    config = config_from_dict(raw)
    model = build_model(config).load(_Weights(seed), case["dtype"], "cuda:0")
    requests = _requests(case)
    longest = max(held + new for held, new in requests)
    pages = sum(-(-(held + new) // PAGE) + 1 for held, new in requests)
    cached_pages = sum(held // PAGE for held, _new in requests)
    length = -(-longest // PAGE) * PAGE + PAGE
    if case["shape"] == "tiny":
        length = min(length, TINY["max_position_embeddings"])
    runner = Runner(model, build_engine_config(
        dtype=case["dtype"], page_size=PAGE, kv_tokens=(pages + cached_pages + 8) * PAGE, max_running=len(requests),
        max_queue_size=len(requests) + 1, max_model_len=length, token_budget=max(case["budget"], len(requests)),
        prefill_chunk=max(case["budget"], 16), prefix_cache_pages=cached_pages + 8), "cuda:0")
    tokens = _tokens(case, seed, config.vocab_size)
    # the history of the conversations: into the cache, and from there into the prefix index
    for index, ((held, _new), ids) in enumerate(zip(requests, tokens)):
        if held:
            name = f"h{index}"
            runner.cache.admit(name)
            for first in range(0, held, 2048):
                runner.run([StepEntry(name, ids[first:min(held, first + 2048)], first)])
            runner.cache.release(name, ids[:held + 1])
    if runner.graphs is not None and case["steps"]:
        runner.graphs.capture_all()  # (what a server does at its start)
    return {"runner": runner, "tokens": tokens, "held": [held for held, _new in requests], "schedule": _schedule(case)}


def run(state):
    runner, tokens, held = state["runner"], state["tokens"], state["held"]
    names = [f"r{index}" for index in range(len(held))]
    for name, ids, cached in zip(names, tokens, held):
        found = runner.cache.admit(name, ids[:cached + 1] if cached else None)
        assert found == cached
    out = []
    for step in state["schedule"]:
        entries = [StepEntry(names[r], tokens[r][held[r] + first:held[r] + first + count], held[r] + first,
                             (count - 1,) if wanted else ()) for r, first, count, wanted in step]
        logits = runner.run(entries)
        if logits.shape[0]:
            out.append(logits)
    for name in names:
        runner.cache.release(name)
    return out


# ---------------------------------------------------------------- what a pass cannot do without
def _weight_counts(raw, case):
    """(numbers of all matrices but the embedding's and the head's, of the head)."""
    if case["design"] == "qwen2":
        hidden, heads = raw["hidden_size"], raw["num_attention_heads"]
        dim = hidden // heads
        kv = raw["num_key_value_heads"] * dim
        return raw["num_hidden_layers"] * (2 * hidden * hidden + 2 * hidden * kv + 3 * hidden * raw["intermediate_size"]), raw["vocab_size"] * hidden
    width, total = raw["width"], 0
    for layer in raw["layers"]:
        m = layer["mixer"]
        if layer["type"] == "retention":
            total += width * m["heads"] * (2 * m["dim"] + 3 * m["vdim"])
        elif layer["type"] == "latent_attention":
            total += width * (m["heads"] * (m["dim"] + m["rot_dim"] + 2 * m["vdim"]) + m["kv_rank"] + m["rot_dim"])
            total += m["heads"] * m["kv_rank"] * (m["dim"] + m["vdim"])
        else:
            total += 3 * width * m["width"] + 2 * m["width"] * (m["width"] // m["blocks"])
        total += 3 * width * layer["mlp"]["ff"]
    return total, raw["vocab"] * width


def _token_costs(raw, case):
    """(numbers cached per token, flops per token and key that it sees, flops per token of the memories, numbers of
    a request's memories)."""
    if case["design"] == "qwen2":
        dim = raw["hidden_size"] // raw["num_attention_heads"]
        layers = raw["num_hidden_layers"]
        return layers * 2 * raw["num_key_value_heads"] * dim, layers * 4 * raw["num_attention_heads"] * dim, 0, 0
    cached = seen = memory = kept = 0
    for layer in raw["layers"]:
        m = layer["mixer"]
        if layer["type"] == "latent_attention":
            cached += m["kv_rank"] + m["rot_dim"]
            seen += 2 * m["heads"] * (m["dim"] + m["rot_dim"] + m["vdim"])
        elif layer["type"] == "retention":
            memory += 4 * m["heads"] * m["dim"] * m["vdim"]
            kept += m["heads"] * m["dim"] * m["vdim"]
        else:
            memory += 8 * m["width"]
            kept += m["width"] * m["conv"]
    return cached, seen, memory, kept


def work(case):
    """Every step reads the weights once, the cache of its requests once and their memories (read and written, in 32
    bits), and writes its tokens' cache and its logits."""
    raw = _raw(case)
    element = 4 if case["dtype"] == "float32" else 2
    matrices, head = _weight_counts(raw, case)
    cached, seen, memory, kept = _token_costs(raw, case)
    held = [h for h, _new in _requests(case)]
    moved = flops = 0.0
    for step in _schedule(case):
        wanted = sum(want for *_rest, want in step)
        tokens = sum(count for _r, _first, count, _want in step)
        moved += (matrices + (head if wanted else 0)) * element + 2 * tokens * cached * element
        moved += wanted * (raw.get("vocab_size") or raw["vocab"]) * 4 + len(step) * 2 * kept * 4
        flops += 2.0 * tokens * matrices + 2.0 * wanted * head + tokens * memory
        for r, first, count, _want in step:
            moved += (held[r] + first) * cached * element
            flops += seen * (count * (held[r] + first) + count * (count + 1) / 2)
    return {"bytes": moved, "flops": flops}


def tolerance(case):
    """Two right implementations of the same precision differ by what their roundings add up to over the layers: in 16
    bits the same step run twice is up to 0.01 apart (parts of a sum arrive in another order; Polosun: 0.006 from the
    64-bit result), in 32 bits 3e-6 from the 64-bit result."""
    if case["dtype"] == "float32":
        return {"rel": 1.2e-5, "max": 2e-4}
    return {"rel": 0.03 if case["design"] == "qwen2" else 0.02, "max": 0.3}


# ---------------------------------------------------------------- the same in 64 bits
def _rotary(dims, theta, upto, factor=None):
    """cos and sin [positions, dims / 2].  The tables are the model's own and 32 bits wide by its definition (angle =
    position x frequency in 32 bits); everything that is done with them here is done in 64."""
    f = 1.0 / (theta ** (torch.arange(0, dims, 2, dtype=torch.float32) / dims))
    gain = 1.0
    if factor is not None:
        turn = lambda t: dims * math.log(factor["original"] / (2.0 * math.pi * t)) / (2.0 * math.log(theta))  # noqa: E731
        low, high = max(math.floor(turn(factor["fast"])), 0), min(math.ceil(turn(factor["slow"])), dims - 1)
        ramp = ((torch.arange(dims // 2, dtype=torch.float32) - low) / max(high - low, 0.001)).clamp(0.0, 1.0)
        f = f / factor["factor"] * ramp + f * (1.0 - ramp)
        gain = 0.1 * math.log(factor["factor"]) + 1.0
    angles = torch.arange(upto, dtype=torch.float32)[:, None] * f[None, :]
    return (angles.cos() * gain).double().cuda(), (angles.sin() * gain).double().cuda()


def _turn(x, cos, sin):
    """x [T, heads, dim] at positions 0..T-1: number i of the turned part with number i + half of it."""
    n = cos.shape[1]
    c, s = cos[: x.shape[0], None, :], sin[: x.shape[0], None, :]
    u, v = x[..., :n], x[..., n:2 * n]
    return torch.cat([u * c - v * s, v * c + u * s, x[..., 2 * n:]], dim=-1)


def _rms(x, eps):
    return x / torch.sqrt((x * x).mean(dim=-1, keepdim=True) + eps)


def _silu(x):
    return x * torch.sigmoid(x)


def _softmax_attention(q, k, v, scale, group):
    """Causal: q [T, heads, d], k and v [T, heads / group, .]; the queries in pieces."""
    tokens = q.shape[0]
    k, v = k.permute(1, 2, 0), v.permute(1, 0, 2)
    out = []
    for first in range(0, tokens, 512):
        last = min(tokens, first + 512)
        rows = q[first:last].permute(1, 0, 2)
        rows = rows.reshape(k.shape[0], group * (last - first), -1)
        scores = torch.matmul(rows, k[..., :last]) * scale
        hidden = torch.arange(last, device="cuda")[None, :] > torch.arange(first, last, device="cuda")[:, None]
        scores = scores.reshape(k.shape[0], group, last - first, last).masked_fill(hidden, -math.inf)
        mixed = torch.matmul(torch.softmax(scores, dim=-1).reshape(k.shape[0], -1, last), v[:, :last])
        out.append(mixed.reshape(k.shape[0] * group, last - first, -1).permute(1, 0, 2))
    return torch.cat(out).reshape(tokens, -1)


def _exact_qwen2(raw, weight, sequences):
    """The last hidden rows of each of the token sequences, normed."""
    hidden, heads, kv, eps = raw["hidden_size"], raw["num_attention_heads"], raw["num_key_value_heads"], raw["rms_norm_eps"]
    dim, ff, vocab = hidden // heads, raw["intermediate_size"], raw["vocab_size"]
    lengths = [len(s) for s in sequences]
    cos, sin = _rotary(dim, raw["rope_theta"], max(lengths))
    embed = weight("model.embed_tokens.weight", (vocab, hidden))
    x = embed[torch.tensor(sum(sequences, []), device="cuda")].double()
    for i in range(raw["num_hidden_layers"]):
        p = f"model.layers.{i}."
        w = lambda name, *shape: weight(p + name, shape).double()  # noqa: E731, B023
        h = _rms(x, eps) * w("input_layernorm.weight", hidden)
        q, k, v = (h @ w(f"self_attn.{n}_proj.weight", c * dim, hidden).t() + w(f"self_attn.{n}_proj.bias", c * dim)
                   for n, c in (("q", heads), ("k", kv), ("v", kv)))
        mixed = []
        for qs, ks, vs in zip(q.split(lengths), k.split(lengths), v.split(lengths)):
            mixed.append(_softmax_attention(_turn(qs.reshape(-1, heads, dim), cos, sin), _turn(ks.reshape(-1, kv, dim), cos, sin),
                                            vs.reshape(-1, kv, dim), dim ** -0.5, heads // kv))
        x = x + torch.cat(mixed) @ w("self_attn.o_proj.weight", hidden, heads * dim).t()
        h = _rms(x, eps) * w("post_attention_layernorm.weight", hidden)
        gate, up = w("mlp.gate_proj.weight", ff, hidden).t(), w("mlp.up_proj.weight", ff, hidden).t()
        down = w("mlp.down_proj.weight", hidden, ff).t()
        x = x + torch.cat([(_silu(part @ gate) * (part @ up)) @ down for part in h.split(16384)])
    x = _rms(x, eps) * weight("model.norm.weight", (hidden,)).double()
    head = embed if raw["tie_word_embeddings"] else weight("lm_head.weight", (vocab, hidden))
    return x.split(lengths), head


def _exact_polosun(raw, weight, sequences):
    width, vocab, eps = raw["width"], raw["vocab"], raw["norm"]["eps"]
    lengths = [len(s) for s in sequences]
    x = weight("embed", (vocab, width))[torch.tensor(sum(sequences, []), device="cuda")].double()
    left = [x]
    for i, layer in enumerate(raw["layers"]):
        m, p = layer["mixer"], f"l{i}."
        w = lambda name, *shape: weight(p + name, shape).double()  # noqa: E731, B023
        h = _rms(x, eps) * w("norm1")
        if layer["type"] == "retention":
            n, d, vd = m["heads"], m["dim"], m["vdim"]
            cos, sin = _rotary(d, m["rot"]["base"], max(lengths))
            decay = torch.tensor(m["decay"], dtype=torch.float64, device="cuda").log()
            q, k, v = h @ w("mix.q", n * d, width).t(), h @ w("mix.k", n * d, width).t(), h @ w("mix.v", n * vd, width).t()
            mixed = []
            for qs, ks, vs in zip(q.split(lengths), k.split(lengths), v.split(lengths)):
                qs, ks = (_turn(t.reshape(-1, n, d), cos, sin).permute(1, 0, 2) for t in (qs, ks))
                at = torch.arange(qs.shape[1], dtype=torch.float64, device="cuda")
                apart = at[:, None] - at[None, :]
                fade = torch.where(apart >= 0, torch.exp(apart.clamp(min=0) * decay[:, None, None]), 0.0)
                o = torch.matmul(torch.matmul(qs, ks.transpose(1, 2)) * d ** -0.5 * fade, vs.reshape(-1, n, vd).permute(1, 0, 2))
                mixed.append(_rms(o, eps).permute(1, 0, 2).reshape(-1, n * vd))
            branch = (torch.cat(mixed) * _silu(h @ w("mix.g", n * vd, width).t())) @ w("mix.o", width, n * vd).t()
        elif layer["type"] == "latent_attention":
            n, d, r, vd, rank = m["heads"], m["dim"], m["rot_dim"], m["vdim"], m["kv_rank"]
            cos, sin = _rotary(r, m["rot"]["base"], max(lengths), m["rot"]["scaling"])
            q, down = h @ w("mix.q", n * (d + r), width).t(), h @ w("mix.dkv", rank + r, width).t()
            latent = _rms(down[:, :rank], eps) * w("mix.dkv.norm", rank)
            k, v = latent @ w("mix.uk", n * d, rank).t(), latent @ w("mix.uv", n * vd, rank).t()
            mixed = []
            for qs, ks, vs, ds in zip(q.split(lengths), k.split(lengths), v.split(lengths), down.split(lengths)):
                qs, ks = qs.reshape(-1, n, d + r), ks.reshape(-1, n, d)
                shared = _turn(ds[:, None, rank:], cos, sin).expand(-1, n, -1)
                qs = torch.cat([qs[..., :d], _turn(qs[..., d:], cos, sin)], dim=-1)
                mixed.append(_softmax_attention(qs, torch.cat([ks, shared], dim=-1), vs.reshape(-1, n, vd), m["scale"], 1))
            branch = (torch.cat(mixed) * torch.sigmoid(h @ w("mix.g", n * vd, width).t())) @ w("mix.o", width, n * vd).t()
        else:
            size, blocks, taps = m["width"], m["blocks"], m["conv"]
            per = size // blocks
            y = torch.nn.functional.gelu(h @ w("mix.y", size, width).t() + w("mix.y.b", size), approximate="tanh")
            inputs = h @ w("mix.x", size, width).t() + w("mix.x.b", size)
            conv = w("mix.conv", size, taps)
            u = torch.cat([sum(torch.nn.functional.pad(part, (0, 0, taps - 1, 0))[j:j + part.shape[0]] * conv[:, j]
                               for j in range(taps)) for part in inputs.split(lengths)]) + w("mix.conv.b", size)
            gates = [torch.sigmoid(torch.einsum("tbi,boi->tbo", u.reshape(-1, blocks, per), w(f"mix.{g}", blocks, per, per))
                                   + w(f"mix.{g}.b", blocks, per)).reshape(-1, size) for g in ("ra", "ri")]
            a = torch.exp(-8.0 * gates[0] * torch.nn.functional.softplus(w("mix.lam", size)))
            add, mixed = torch.sqrt(1.0 - a * a) * gates[1] * u, []
            for fades, adds in zip(a.split(lengths), add.split(lengths)):
                state, rows = torch.zeros(size, dtype=torch.float64, device="cuda"), torch.empty_like(adds)
                for t in range(adds.shape[0]):
                    state = torch.addcmul(adds[t], fades[t], state, out=rows[t])
                mixed.append(rows)
            branch = (torch.cat(mixed) * y) @ w("mix.o", width, size).t()
        ff = layer["mlp"]["ff"]
        h = _rms(x, eps) * w("norm2")
        branch = branch + (_silu(h @ w("mlp.gate", ff, width).t()) * (h @ w("mlp.up", ff, width).t())) @ w("mlp.down", width, ff).t()
        left.append(x + raw["residual_mult"] * branch)
        average = w("dwa", i + 2)
        x = sum(average[j] * rows for j, rows in enumerate(left))
    return (_rms(x, eps) * weight("final.norm", ()).double()).split(lengths), weight("head", (vocab, width))


def exact(case, seed):
    raw = _raw(case)
    requests = _requests(case)
    if work(case)["flops"] + sum(held for held, _new in requests) * 2.0 * _weight_counts(raw, case)[0] > 5e14:
        return None  # (more than some twenty seconds of 64-bit products)
    sequences = _tokens(case, seed, raw.get("vocab_size") or raw["vocab"])
    weight = lambda name, shape: _tensor(name, shape, seed, case["dtype"])  # noqa: E731
    with torch.no_grad():
        rows, head = (_exact_qwen2 if case["design"] == "qwen2" else _exact_polosun)(raw, weight, sequences)
        head, out = head.double().t(), []
        for step in _schedule(case):
            wanted = [rows[r][requests[r][0] + first + count - 1] for r, first, count, want in step if want]
            if wanted:
                out.append(torch.stack(wanted) @ head)
    return out
