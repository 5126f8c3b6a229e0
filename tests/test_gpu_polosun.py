"""GPU: the Polosun decoder in the engine against the plain implementation (tests/plain_polosun.py): every
mechanism alone, every way of cutting and batching the same requests, reused pages and slots, long prompts and long
decoding, other sizes, and greedy generation through the engine's own entry point."""

from __future__ import annotations

import math
import random

import numpy as np
import pytest
import torch

import plain_polosun
import polosun_util as pu
import replay_util
from conftest import random_tokens

pytestmark = pytest.mark.gpu

# a row's error is the root mean square of the difference of its logits, mean taken off, as a share of the
# logits' own spread.  float32: sums in another order; this is the sharp test of cache, state and batching.
# bfloat16: activations rounded to 8 bits between kernels, with these bold weights (peaked softmax, branches
# weighed up to 1.25) a few per cent at the worst row and under two on average (RMS_LIMIT).
LIMIT = {"float32": 2e-5, "bfloat16": 8e-2}
RMS_LIMIT = {"float32": 1e-5, "bfloat16": 3e-2}


def plain_all(raw, weights, requests):
    return {rid: plain_polosun.forward(raw, weights, tokens).float() for rid, tokens in requests.items()}


def run_and_compare(raw, weights, requests, steps, dtype, plain, page_size=16, max_running=4, limit=None):
    pool = max(replay_util.max_live_tokens(steps, page=page_size), page_size)
    runner = pu.make_runner(raw, weights, dtype, pool, page_size, max_running)
    rows = replay_util.by_position(steps, replay_util.drive_runner(runner, steps))
    for rid in requests:
        assert rid in rows, f"{rid}: no logits"
    worst, rms = pu.spread(rows, plain)
    assert worst <= (limit or LIMIT[dtype]) and rms <= RMS_LIMIT[dtype], (dtype, worst, rms)
    assert runner.cache.stats().slots_used == 0 and runner.cache.stats().pages_used == 0
    return rows


MECHANISMS = {
    "latent_attention": {"type": "latent_attention", "mlp": None,
                         "mixer": {"heads": 2, "dim": 8, "rot_dim": 8, "vdim": 12, "kv_rank": 20, "scale": 0.7,
                                   "rot": {"base": 200.0, "dims": 8}}},
    "latent_attention_stretched": {"type": "latent_attention", "mlp": None,
                                   "mixer": {"heads": 4, "dim": 12, "rot_dim": 16, "vdim": 4, "kv_rank": 8, "scale": 0.5,
                                             "rot": {"base": 1000.0, "dims": 16, "scaling":
                                                     {"factor": 8.0, "fast": 8.0, "original": 32, "slow": 0.5}}}},
    "latent_attention_unturned": {"type": "latent_attention", "mlp": None,
                                  "mixer": {"heads": 2, "dim": 8, "rot_dim": 4, "vdim": 8, "kv_rank": 12, "scale": 0.9}},
    "retention": {"type": "retention", "mlp": None,
                  "mixer": {"heads": 2, "dim": 12, "vdim": 20, "decay": [0.875, 0.99609375], "rot": {"base": 300.0, "dims": 12}}},
    "retention_part_turned": {"type": "retention", "mlp": None,
                              "mixer": {"heads": 3, "dim": 40, "vdim": 8, "decay": [0.5, 0.9, 0.999], "rot": {"base": 20.0, "dims": 6}}},
    "retention_unturned": {"type": "retention", "mlp": None, "mixer": {"heads": 1, "dim": 4, "vdim": 72, "decay": [0.96875]}},
    "rglru": {"type": "rglru", "mlp": None, "mixer": {"width": 40, "blocks": 5, "conv": 3}},
    "rglru_one_tap": {"type": "rglru", "mlp": None, "mixer": {"width": 16, "blocks": 1, "conv": 1}},
    "rglru_long_taps": {"type": "rglru", "mlp": None, "mixer": {"width": 24, "blocks": 2, "conv": 7}},
    "feed_forward": {"type": "rglru", "mlp": {"kind": "dense", "ff": 44}, "mixer": {"width": 8, "blocks": 1, "conv": 2}},
}


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("name", sorted(MECHANISMS))
def test_a_mechanism_alone(name, dtype):
    """One layer of one kind: whole prompts, then the same tokens in portions down to two tokens and one by one
    (shorter than the convolution's reach, across pages), two requests side by side."""
    raw = pu.single(MECHANISMS[name])
    weights = pu.make_weights(raw, seed=3)
    requests = {"a": random_tokens(45, raw["vocab"], 1), "b": random_tokens(21, raw["vocab"], 2), "c": [7]}
    plain = plain_all(raw, weights, requests)
    run_and_compare(raw, weights, requests, replay_util.whole(requests), dtype, plain)
    run_and_compare(raw, weights, requests, replay_util.portions(requests, sizes=(2, 3, 2, 17, 2, 5)), dtype, plain)
    run_and_compare(raw, weights, requests, replay_util.mixed(requests, live=3, chunk_sizes=(2, 7, 3), decode_tail=9),
                    dtype, plain, max_running=3)


SCHEDULES = {
    "whole": replay_util.whole,
    "tail": lambda requests: replay_util.tail_one_by_one(requests, tail=20),
    "portions": replay_util.portions,
    "mixed": lambda requests: replay_util.mixed(requests, live=4),
}
LENGTHS = {"A": [5, 17, 33, 70, 100, 1], "B": [2, 9, 40, 64, 131]}


@pytest.fixture(scope="module")
def models():
    out = {}
    for index, (name, raw) in enumerate(pu.SMALL.items()):
        weights = pu.make_weights(raw, seed=20 + index)
        requests = {f"{name}{i}": random_tokens(n, raw["vocab"], seed=50 + i) for i, n in enumerate(LENGTHS[name])}
        out[name] = (raw, weights, requests, plain_all(raw, weights, requests))
    return out


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("schedule", sorted(SCHEDULES))
@pytest.mark.parametrize("name", sorted(pu.SMALL))
def test_logits_do_not_depend_on_cutting_or_batching(models, name, schedule, dtype):
    """Prefill against token-by-token decoding, portions of several sizes, unequal requests in one batch against
    each alone; six requests take turns on four slots, and the pool is no larger than the schedule's peak."""
    raw, weights, requests, plain = models[name]
    run_and_compare(raw, weights, requests, SCHEDULES[schedule](requests), dtype, plain)


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("name", sorted(pu.SMALL))
def test_captured_steps_give_the_same_logits(models, name, dtype):
    """Steps of single tokens replay captured graphs (and short mixed steps theirs, from the second time a shape
    comes), with uncaptured steps between the replays: every replay is checked against the plain logits, and states
    move on once per token although a capture runs the kernels on rows of padding."""
    raw, weights, requests, plain = models[name]
    steps = replay_util.fixed_portions(requests, portion=8, live=3, decode_tail=14)
    pool = max(replay_util.max_live_tokens(steps, page=16), 16)
    runner = pu.make_runner(raw, weights, dtype, pool, 16, 4, graph_decode=True)
    assert runner.graphs is not None, "the model's parts all say that they may be captured"
    rows = replay_util.by_position(steps, replay_util.drive_runner(runner, steps))
    worst, rms = pu.spread(rows, plain)
    assert runner.graph_replays >= 10 and runner.mixed_graph_replays > 0, (runner.graph_replays, runner.mixed_graph_replays)
    assert worst <= LIMIT[dtype] and rms <= RMS_LIMIT[dtype], (worst, rms)


@pytest.mark.parametrize("page_size", [4, 64])
def test_other_page_sizes(models, page_size):
    raw, weights, requests, plain = models["A"]
    run_and_compare(raw, weights, requests, replay_util.mixed(requests, live=3, seed=5), "float32", plain,
                    page_size=page_size, max_running=3)


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
def test_random_traces_reuse_pages_and_slots(models, dtype):
    """Random cuts (one token, two, up to a page's edge, one past it) of ten requests on three slots: every slot
    and page is handed out again, and a state that a new request found uncleared would show at its first token."""
    raw, weights, _, _ = models["B"]
    rng = random.Random(4)
    requests, steps = replay_util.random_trace(rng, [3, 40, 17, 1, 33, 64, 2, 18, 49, 31], raw["vocab"], 16, live_most=3)
    plain = plain_all(raw, weights, requests)
    wanted = {rid: {pos: None for pos in range(len(tokens))} for rid, tokens in requests.items()}
    pool = max(replay_util.max_live_tokens(steps, page=16), 16)
    runner = pu.make_runner(raw, weights, dtype, pool, 16, 3)
    rows = replay_util.by_position(steps, replay_util.drive_runner(runner, steps))
    assert set(rows) <= set(wanted) and rows
    worst, _ = pu.spread(rows, plain)
    assert worst <= LIMIT[dtype], worst


NEEDLE, ASK, FILLERS = 1, 2, 40  # token ids: the one to be found, the one that looks for it, the first of the rest


def planted(kind: str):
    """A single layer whose weights are changed by hand so that one score stands out: the token ASK looks, through a
    query dimension that only it has, for a key dimension that only the token NEEDLE has, wherever that lies."""
    if kind == "latent_attention":
        layer = {"type": "latent_attention", "mlp": None,
                 "mixer": {"heads": 2, "dim": 16, "rot_dim": 8, "vdim": 16, "kv_rank": 24, "scale": 0.25,
                           "rot": {"base": 10000.0, "dims": 8}}}
    else:
        layer = {"type": "retention", "mlp": None,
                 "mixer": {"heads": 2, "dim": 16, "vdim": 16, "decay": [0.998046875, 0.9990234375],
                           "rot": {"base": 10000.0, "dims": 8}}}
    raw = pu.single(layer, width=32, vocab=64)
    w = pu.make_weights(raw, seed=9)
    w["embed"][:, 0:2] = 0.0
    w["embed"][NEEDLE, 0] = 8.0
    w["embed"][ASK, 1] = 8.0
    heads, dim = layer["mixer"]["heads"], layer["mixer"]["dim"]
    if kind == "latent_attention":
        per = dim + layer["mixer"]["rot_dim"]
        w["l0.mix.dkv"][:, 0:2] = 0.0
        w["l0.mix.dkv"][0, :] = 0.0
        w["l0.mix.dkv"][0, 0] = 4.0            # latent 0 is the needle's mark
        w["l0.mix.uk"][:, 0] = 0.0
        w["l0.mix.q"][:, 0:2] = 0.0
        for h in range(heads):
            w["l0.mix.uk"][h * dim, :] = 0.0
            w["l0.mix.uk"][h * dim, 0] = 4.0    # plain key dimension 0 of every head reads it
            w["l0.mix.q"][h * per, :] = 0.0
            w["l0.mix.q"][h * per, 1] = 4.0     # plain query dimension 0 of every head reads the asker's mark
    else:
        at = 12                                 # a dimension that does not turn
        for name, column in (("k", 0), ("q", 1)):
            w["l0.mix." + name][:, 0:2] = 0.0
            for h in range(heads):
                w["l0.mix." + name][h * dim + at, :] = 0.0
                w["l0.mix." + name][h * dim + at, column] = 16.0
    w["l0.mix.o"] *= 4.0                        # the layer's branch outweighs the embedding's own share of the logits
    return raw, {k: v.to(torch.bfloat16).float() for k, v in w.items()}


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("kind", ["latent_attention", "retention"])
def test_one_key_among_hundreds_is_found_wherever_it_lies(kind, dtype):
    """The needle at the first positions, at page borders, far back; asked for inside a prompt's portion and by a
    token decoded alone, across several requests that share a pool and reuse slots.  A lost key, a key of a wrong
    page or slot, or a state that is not carried moves these logits by far more than the tolerance (checked below
    on the plain implementation itself)."""
    raw, weights = planted(kind)
    length = 600
    places = [0, 1, 15, 16, 17, 63, 64, 300, 511, 512, 590]
    requests = {}
    for place in places:
        tokens = [FILLERS + t % (raw["vocab"] - FILLERS) for t in random_tokens(length, 1000, 30 + place)]
        tokens[place] = NEEDLE
        requests[f"n{place}"] = tokens + [ASK, FILLERS, ASK]
    plain = plain_all(raw, weights, requests)
    # the test of the test: without the needle the asked rows are far off
    for rid in ("n0", "n300"):
        blind = list(requests[rid])
        blind[blind.index(NEEDLE)] = FILLERS + 3
        other = plain_polosun.forward(raw, weights, blind).float()
        for row in (length, length + 2):
            diff = other[row] - plain[rid][row]
            assert float((diff - diff.mean()).pow(2).mean().sqrt() / plain[rid][row].std()) > 0.5
    steps, sizes = [], (129, 2, 255, 31, 64, 3)
    waiting = list(requests.items())
    while waiting:
        pair = [waiting.pop(0) for _ in range(min(2, len(waiting)))]
        fed = {rid: 0 for rid, _ in pair}
        turn = 0
        while any(fed[rid] < len(tokens) for rid, tokens in pair):
            entries, end = [], []
            for index, (rid, tokens) in enumerate(pair):
                left = len(tokens) - fed[rid]
                if left == 0:
                    continue
                # the last token (an asker) comes alone; the asker before it inside a portion
                size = 1 if left == 1 else min(sizes[(turn + index) % len(sizes)], left - 1)
                want = [i for i in range(size) if fed[rid] + i >= length]
                entries.append({"id": rid, "tokens": tokens[fed[rid]: fed[rid] + size], "want": want})
                fed[rid] += size
                if fed[rid] == len(tokens):
                    end.append(rid)
            turn += 1
            steps.append({"step": len(steps), "entries": entries, "end": end})
    pool = replay_util.max_live_tokens(steps, page=16)
    runner = pu.make_runner(raw, weights, dtype, pool, 16, 2)
    rows = replay_util.by_position(steps, replay_util.drive_runner(runner, steps))
    assert all(sorted(rows[rid]) == [length, length + 1, length + 2] for rid in requests)
    worst, _ = pu.spread(rows, plain)
    assert worst <= LIMIT[dtype], worst


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
def test_long_decoding(dtype):
    """A prompt of 300 tokens, then 250 tokens decoded one by one across page borders, every layer kind in the model."""
    raw = pu.SMALL_A
    weights = pu.make_weights(raw, seed=31)
    requests = {"long": random_tokens(550, raw["vocab"], 7)}
    stepper = plain_polosun.Stepper(raw, weights)
    plain = {"long": torch.stack([stepper.token(t) for t in requests["long"]]).float()}
    steps = replay_util.tail_one_by_one(requests, tail=250)
    run_and_compare(raw, weights, requests, steps, dtype, plain, max_running=1)


def test_greedy_generation_through_the_engine(models):
    """The engine's own entry point and scheduler (prompts in portions, several requests at once) generate what the
    plain implementation generates."""
    from cie_amd import Engine, GenerationConfig
    from cie_amd.config import config_from_dict

    raw, weights, _, _ = models["A"]
    prompts = [random_tokens(n, raw["vocab"], 80 + n) for n in (3, 19, 42)]
    for dtype in ("float32", "bfloat16"):
        engine = Engine(config=config_from_dict(raw), seed=0, dtype=dtype, page_size=16, kv_tokens=512, max_running=3,
                        max_model_len=128, prefill_chunk=8, token_budget=24, prefix_cache_pages=0)
        engine.model.load(pu.Fixed(weights), dtype, "cuda:0")
        results = engine.generate(prompts, GenerationConfig(max_output_tokens=12))
        for prompt, result in zip(prompts, results):
            assert len(result.token_ids) == 12
            turned = replay_util.greedy_tokens_follow_plain(
                lambda tokens: plain_polosun.forward(raw, weights, tokens), prompt, result.token_ids,
                (lambda tokens: plain_polosun.forward(raw, weights, tokens, dtype=torch.bfloat16)) if dtype == "bfloat16" else None)
            assert turned <= (0 if dtype == "float32" else 3)


def test_the_trace_runner_replays_a_model_folder(tmp_path, models):
    """bin/trace_run on a folder written for it: same logits as the plain implementation, four slots by default."""
    import json
    import subprocess
    import sys

    from cie_amd.weights import write_tensors
    from conftest import ROOT

    raw, weights, requests, plain = models["B"]
    folder = write_tensors(tmp_path / "model", raw, {k: v.to(torch.bfloat16) for k, v in weights.items()})
    steps = replay_util.mixed(requests, live=4)
    out = tmp_path / "out"
    pool = replay_util.max_live_tokens(steps, page=64)
    done = subprocess.run([sys.executable, str(ROOT / "bin" / "trace_run"), "--model", str(folder), "--dtype", "float32",
                           "--out", str(out), "--max-tokens", str(pool)],
                          input="\n".join(json.dumps(s) for s in steps) + "\n", capture_output=True, text=True, timeout=600)
    assert done.returncode == 0, done.stderr[-2000:]
    assert [line for line in done.stdout.split("\n") if line.startswith("done")] == [f"done {s['step']}" for s in steps]
    outputs = {s["step"]: np.fromfile(out / f"{s['step']}.f32", dtype="<f4").reshape(-1, raw["vocab"])
               for s in steps if any(e["want"] for e in s["entries"])}
    worst, _ = pu.spread(replay_util.by_position(steps, outputs), plain)
    assert worst <= LIMIT["float32"], worst


# ---------------------------------------------------------------- kernels alone
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("rows", [1, 7, 16, 17, 64, 150])
def test_block_diagonal_product_in_all_its_forms(rows, dtype):
    """Few rows, tiles, and (bfloat16) the matrix cores; blocks read from and written to columns of wider rows, with
    bias, with a sigmoid gate, float32 results from bfloat16 operands; a K that is no multiple of 32, and one that is
    no multiple of 8 (which keeps off the matrix cores)."""
    from cie_amd.kernels import ops

    g = torch.Generator().manual_seed(rows)
    for blocks, n, k, a_block, extra in ((3, 24, 40, 56, 8), (2, 80, 96, 96, 0), (5, 17, 12, 20, 4)):
        a = torch.randn(rows, extra + (blocks - 1) * a_block + k + 3, generator=g).to(dtype).cuda()
        w = (torch.randn(blocks, n, k, generator=g) / k ** 0.5).to(dtype).cuda()
        bias = torch.randn(blocks, n, generator=g).to(dtype).cuda()
        gate = torch.randn(rows, 5 + blocks * n, generator=g).to(dtype).cuda()
        picked = torch.stack([a[:, extra + b * a_block: extra + b * a_block + k] for b in range(blocks)], 1).double()
        plain = torch.einsum("mbk,bnk->mbn", picked, w.double())
        tol = 2e-5 if dtype == torch.float32 else 2e-2
        out = ops.block_linear(a, w, a_block=a_block, a_offset=extra, out_dtype=torch.float32)
        assert torch.allclose(out.double().reshape(rows, blocks, n), plain, atol=2e-5 if dtype == torch.float32 else 1e-4)
        with_bias = ops.block_linear(a, w, bias, a_block=a_block, a_offset=extra)
        assert with_bias.dtype == dtype
        assert torch.allclose(with_bias.double().reshape(rows, blocks, n), plain + bias.double(), atol=tol, rtol=tol)
        wide = torch.full((rows, 6 + blocks * (n + 2)), 7.0, dtype=dtype, device="cuda")
        ops.block_linear(a, w, a_block=a_block, a_offset=extra, out=wide, out_offset=6, c_block=n + 2, gate=gate, gate_offset=5)
        gated = plain * torch.sigmoid(gate[:, 5:].double().reshape(rows, blocks, n))
        got = wide[:, 6:].reshape(rows, blocks, n + 2)
        assert torch.allclose(got[:, :, :n].double(), gated, atol=tol, rtol=tol)
        assert bool((wide[:, :6] == 7).all()) and bool((got[:, :-1, n:] == 7).all())  # nothing beside the blocks is touched
    # a row's result does not depend on the rows beside it
    if 1 < rows <= 4 or (dtype == torch.float32 and rows <= 16):  # (within one form of the kernel, bit for bit)
        alone = ops.block_linear(a[:1].contiguous(), w, a_block=a_block, a_offset=extra, out_dtype=torch.float32)
        assert torch.equal(alone, out[:1])


@pytest.mark.parametrize("rows", [5, 16, 17, 64, 65, 520, 600])
@pytest.mark.parametrize("blocks,n,k", [(1, 16, 8), (3, 72, 40), (2, 130, 128), (2, 64, 136), (5, 24, 256), (1, 200, 264)])
def test_block_diagonal_product_on_the_matrix_cores(rows, blocks, n, k):
    """Operands that take them: one tile of 16 rows and tiles of 64, fewer and more blocks of rows than XCDs; one group of
    8 k, K inside a round of four slices, one round, one group more, two rounds and one group more."""
    from cie_amd.kernels import ops

    g = torch.Generator().manual_seed(rows + k)
    a_block = k + 16
    a = torch.randn(rows, 8 + blocks * a_block, generator=g).bfloat16().cuda()
    w = (torch.randn(blocks, n, k, generator=g) / k ** 0.5).bfloat16().cuda()
    bias = torch.randn(blocks, n, generator=g).bfloat16().cuda()
    gate = torch.randn(rows, blocks * n, generator=g).bfloat16().cuda()
    picked = torch.stack([a[:, 8 + b * a_block: 8 + b * a_block + k] for b in range(blocks)], 1).cpu().double()
    plain = torch.stack([picked[:, b] @ w[b].cpu().double().t() for b in range(blocks)], 1)
    size = torch.stack([picked[:, b].abs() @ w[b].cpu().double().abs().t() for b in range(blocks)], 1)
    out = ops.block_linear(a, w, a_block=a_block, a_offset=8, out_dtype=torch.float32).cpu().double().reshape(rows, blocks, n)
    # exact products of bfloat16 numbers, k float32 sums: each rounds by at most 2^-24 of what it has summed
    assert torch.all((out - plain).abs() <= k * 2.0 ** -24 * size)
    wide = torch.full((rows, 8 + blocks * (n + 8)), 7.0, dtype=torch.bfloat16, device="cuda")
    ops.block_linear(a, w, bias, a_block=a_block, a_offset=8, out=wide, out_offset=8, c_block=n + 8, gate=gate)
    gated = (plain + bias.cpu().double()) * torch.sigmoid(gate.cpu().double().reshape(rows, blocks, n))
    got = wide[:, 8:].cpu().double().reshape(rows, blocks, n + 8)
    assert torch.all((got[:, :, :n] - gated).abs() <= 2.0 ** -8 * gated.abs() + 1e-5 * (size + 1))  # (rounded once)
    assert bool((wide[:, :8] == 7).all()) and bool((got[:, :, n:] == 7).all())



@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_layer_boundary_kernel(dtype):
    from cie_amd.kernels import ops

    g = torch.Generator().manual_seed(1)
    for rows, hidden in ((3, 40), (130, 1024), (9, 2048)):
        history = torch.randn(5, rows, hidden, generator=g).cuda()
        x = torch.randn(rows, hidden, generator=g).cuda()
        a = torch.randn(rows, hidden, generator=g).to(dtype).cuda()
        b = torch.randn(rows, hidden, generator=g).to(dtype).cuda()
        weights = torch.randn(4, generator=g).cuda()
        kept = history.clone()
        stream, normed = ops.depth_stream(x, a, b, mult=0.7, history=history, newest=3, weights=weights, gains=(1.5, 0.25),
                                          out_dtype=dtype, eps=1e-5)
        new = x.double() + 0.7 * (a.double() + b.double())
        assert torch.allclose(history[3].double(), new, atol=1e-5) and torch.equal(history[[0, 1, 2, 4]], kept[[0, 1, 2, 4]])
        want = sum(weights[j].double() * (new if j == 3 else kept[j].double()) for j in range(4))
        assert torch.allclose(stream.double(), want, atol=2e-5)
        unit = want / torch.sqrt((want * want).mean(-1, keepdim=True) + 1e-5)
        tol = 1e-5 if dtype == torch.float32 else 2e-2
        assert torch.allclose(normed[0].double(), unit * 1.5, atol=tol, rtol=tol)
        assert torch.allclose(normed[1].double(), unit * 0.25, atol=tol, rtol=tol)
        # one branch, no average, one norm; and norms alone
        stream, normed = ops.depth_stream(x, a, mult=2.0, gains=(1.0,), out_dtype=dtype, eps=1e-5)
        assert torch.allclose(stream.double(), x.double() + 2.0 * a.double(), atol=1e-5) and len(normed) == 1
        nothing, normed = ops.depth_stream(x, gains=(3.0, 1.0), out_dtype=dtype, eps=1e-5, want_stream=False)
        unit = x.double() / torch.sqrt((x.double() ** 2).mean(-1, keepdim=True) + 1e-5)
        assert nothing is None and torch.allclose(normed[0].double(), 3.0 * unit, atol=tol, rtol=tol)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("rows,hidden,terms,newest", [
    (1, 4, 1, 0), (5, 2048, 9, 8), (5, 2048, 8, 3), (3, 4096, 10, 9), (2, 4100, 17, 16), (2, 6144, 18, 0), (4, 260, 3, 4)])
def test_layer_boundary_kernel_over_depths_and_widths(dtype, rows, hidden, terms, newest):
    """The boundary with four numbers a thread: one piece and several a thread, a width that ends inside a wave, up to
    eight earlier rows asked for at once and more, the row just made first, in the middle, last and outside the average;
    and the same over views that start off a 16-byte line, which take the form of single numbers."""
    from cie_amd.kernels import ops

    g = torch.Generator().manual_seed(2)
    layers = max(terms, newest + 1)
    weights = torch.randn(terms, generator=g)
    for shift, n_parts in ((0, 0), (1, 0), (0, 1), (0, 9), (1, 3)):
        def rand(*shape, kind=torch.float32):  # (a tensor whose first number lies `shift` numbers off the allocation's start)
            n = torch.Size(shape).numel()
            return torch.randn(n + shift, generator=g).to(kind).cuda()[shift:].view(shape)
        history, x = rand(layers, rows, hidden), rand(rows, hidden)
        a, b = rand(rows, hidden, kind=dtype), rand(rows, hidden, kind=dtype)
        parts = rand(n_parts, rows, hidden) if n_parts else None  # (a branch that comes as the parts of a product)
        kept = history.clone()
        stream, normed = ops.depth_stream(x, a, b, mult=0.7, history=history, newest=newest, weights=weights.cuda(),
                                          gains=(1.5, 0.25), out_dtype=dtype, eps=1e-5, parts=parts)
        new = x.double() + 0.7 * (a.double() + b.double() + (parts.double().sum(0) if n_parts else 0.0))
        rest = [j for j in range(layers) if j != newest]
        assert torch.allclose(history[newest].double(), new, atol=1e-5) and torch.equal(history[rest], kept[rest])
        parts = [weights[j].double().item() * (new if j == newest else kept[j].double()) for j in range(terms)]
        want, size = sum(parts), sum(p.abs() for p in parts)
        # each of the sum's `terms` roundings is at most half a unit in the last place of a partial sum below `size`; three
        # more, and one a part, make the row just made, whose own partial sums stay below 64
        assert torch.all((stream.double() - want).abs() <= 2.0 ** -24 * ((terms + 3) * (size + 2.0) + n_parts * 64.0))
        unit = want / torch.sqrt((want * want).mean(-1, keepdim=True) + 1e-5)
        tol = 1e-5 if dtype == torch.float32 else 2e-2
        assert torch.allclose(normed[0].double(), unit * 1.5, atol=tol, rtol=tol)
        assert torch.allclose(normed[1].double(), unit * 0.25, atol=tol, rtol=tol)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("rows,n_parts", [(3, 1), (5, 7), (5, 8), (128, 9), (129, 4), (130, 5), (2, 16)])
def test_layer_boundary_kernel_that_sums_a_branch_in_parts(dtype, rows, n_parts):
    """One branch and the parts of another, as a layer whose down product was cut leaves them: as many parts as are asked
    for at once, one more and one less, in the forms for few rows and for many; the bits of the parts added in order."""
    from cie_amd.kernels import ops

    g = torch.Generator().manual_seed(5)
    hidden = 264
    x, a = torch.randn(rows, hidden, generator=g).cuda(), torch.randn(rows, hidden, generator=g).to(dtype).cuda()
    parts, weights = torch.randn(n_parts, rows, hidden, generator=g).cuda(), torch.randn(3, generator=g).cuda()
    history = torch.randn(3, rows, hidden, generator=g).cuda()
    kept = history.clone()
    stream, normed = ops.depth_stream(x, a, None, mult=0.5, history=history, newest=2, weights=weights, gains=(1.5,), out_dtype=dtype,
                                      eps=1e-5, parts=parts)
    branch = a.float()
    for part in parts:
        branch = branch + part
    assert torch.equal(history[2], x + 0.5 * branch) and torch.equal(history[:2], kept[:2])  # (half of it is exact)
    want = sum(weights[j].double() * history[j].double() for j in range(3))
    # three roundings of half a unit in the last place of sums whose terms stay below 64
    assert torch.all((stream.double() - want).abs() <= 3 * 2.0 ** -24 * 64.0)
    unit = want / torch.sqrt((want * want).mean(-1, keepdim=True) + 1e-5)
    tol = 1e-5 if dtype == torch.float32 else 2e-2
    assert torch.allclose(normed[0].double(), unit * 1.5, atol=tol, rtol=tol)


@pytest.mark.parametrize("captured", [False, True])
def test_a_layer_whose_down_product_comes_in_parts(monkeypatch, captured):
    """A feed-forward wide enough for its down product to be cut (few rows: the streaming kernel's parts; 150 rows: the
    tiles'), against the plain implementation."""
    from cie_amd.parts import linear

    raw = pu.single({"type": "rglru", "mlp": {"kind": "dense", "ff": 4104}, "mixer": {"width": 16, "blocks": 2, "conv": 4}}, width=64)
    weights = pu.make_weights(raw, seed=6)
    requests = {"a": random_tokens(150, raw["vocab"], 1), "b": random_tokens(21, raw["vocab"], 2), "c": [7, 3]}
    plain = plain_all(raw, weights, requests)
    seen, parts_of = [], linear.KParts.__init__
    monkeypatch.setattr(linear.KParts, "__init__", lambda self, parts: (seen.append(parts.shape[:2]), parts_of(self, parts))[1])
    monkeypatch.setattr(linear, "plan_tiles", lambda rows, n, k, most_parts=1, behind=None: (64, 64, 3) if most_parts > 1 and k > 4000 else None)
    steps = replay_util.fixed_portions(requests, portion=150, live=3, decode_tail=8) if captured else replay_util.tail_one_by_one(requests, tail=8)
    pool = max(replay_util.max_live_tokens(steps, page=16), 16)
    runner = pu.make_runner(raw, weights, "bfloat16", pool, 16, 4, graph_decode=captured)
    rows = replay_util.by_position(steps, replay_util.drive_runner(runner, steps))
    worst, rms = pu.spread(rows, plain)
    assert worst <= LIMIT["bfloat16"] and rms <= RMS_LIMIT["bfloat16"], (worst, rms)
    assert any(parts > 1 and count <= 128 for parts, count in seen) and any(parts == 3 and count > 128 for parts, count in seen), seen


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("lengths,channels,taps,segments", [
    ((64, 1, 129), 48, 4, 64), ((63, 65), 16, 4, 64), ((2048,), 128, 4, 64), ((2049, 70), 40, 3, 64), ((4100,), 16, 4, 64),
    ((300, 5), 24, 4, 2), ((97,), 40, 4, 16), ((9, 2, 3), 72, 4, 1)])
def test_gated_recurrence_and_its_convolution(dtype, lengths, channels, taps, segments):
    """Stretches of one token and of the most a round has, portions one short of a round, one round, and one longer than
    it, fewer tokens than stretches, workgroups that end behind the last channel; against the walk in order in 64 bits."""
    from cie_amd.kernels import ops

    g = torch.Generator().manual_seed(3)
    tokens, width = sum(lengths), channels // 2
    slots = list(range(len(lengths)))[::-1]
    proj = torch.randn(tokens, 2 * channels, generator=g).to(dtype).cuda()
    y_pre, x_in = proj[:, :channels], proj[:, channels:]
    taps_w = torch.randn(channels, taps, generator=g).to(dtype).cuda()
    bias = torch.randn(channels, generator=g).to(dtype).cuda()
    past = torch.randn(len(lengths), taps - 1, channels, generator=g).cuda()
    state = torch.randn(len(lengths), channels, generator=g).cuda()
    gates = torch.randn(tokens, 2 * channels, generator=g).cuda()
    rate = -8.0 * torch.rand(channels, generator=g).cuda()
    starts = [sum(lengths[:i]) for i in range(len(lengths) + 1)]
    meta = lambda values: torch.tensor(values, dtype=torch.int32).cuda()
    of_token = meta([i for i, n in enumerate(lengths) for _ in range(n)])
    old_past, old_state = past.clone(), state.clone()
    u = ops.causal_conv(x_in, taps_w, bias, past, of_token, meta(slots), meta(starts))
    out = ops.gated_recurrence(y_pre, x_in, u, gates, width, rate, state, past, meta(slots), meta(starts), len(lengths),
                               taps, segments)
    # a bfloat16 result is rounded once; float32 sums of up to 17 and of some ten terms in front of it
    tol = dict(atol=3e-5, rtol=3e-5) if dtype == torch.float32 else dict(atol=3e-5, rtol=2.0 ** -8)
    for i, n in enumerate(lengths):
        at, slot = starts[i], slots[i]
        series = torch.cat([old_past[slot], x_in[at: at + n].float()])
        window = series.double().unfold(0, taps, 1)  # [n, channels, taps]
        conv = (window * taps_w.double()).sum(-1) + bias.double()
        assert torch.allclose(u[at: at + n].double(), conv, **tol)
        assert torch.equal(past[slot], series[-(taps - 1):])
        gate = gates[at: at + n].double().view(n, 2, 2, width).cpu()
        log_a = rate.double().cpu() * torch.sigmoid(gate[:, :, 0].reshape(n, channels))
        moved = torch.sqrt(-torch.expm1(2 * log_a)) * torch.sigmoid(gate[:, :, 1].reshape(n, channels)) * u[at: at + n].double().cpu()
        S, walked = old_state[slot].double().cpu(), []
        for t in range(n):
            S = torch.exp(log_a[t]) * S + moved[t]
            walked.append(S)
        want = torch.stack(walked) * torch.nn.functional.gelu(y_pre[at: at + n].double().cpu(), approximate="tanh")
        # (S fades by 1 - a^2 against what it takes in: its float32 roundings do not add up over the tokens)
        assert torch.allclose(out[at: at + n].double().cpu(), want, **tol)
        assert torch.allclose(state[slot].double().cpu(), S, atol=3e-5, rtol=3e-5)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("lengths,heads,dim,vdim,span", [
    ((33,), 2, 40, 24, 1), ((70, 5, 129), 1, 128, 128, 1), ((64, 31), 2, 160, 72, 2), ((200,), 3, 16, 256, 1),
    ((1, 1, 1), 2, 128, 128, 1), ((1, 2), 4, 16, 16, 4), ((40,), 2, 24, 136, 2)])
def test_retention_over_the_edges_of_its_pieces(dtype, lengths, heads, dim, vdim, span):
    """Blocks that end inside their 32 tokens, heads of fewer and of more pieces than one round of loads, columns in one
    panel and two, norms over one lane's column, over four and over more; both walks; against 64 bits token by token."""
    from cie_amd.kernels import ops

    g = torch.Generator().manual_seed(4)
    tokens, slots = sum(lengths), list(range(len(lengths)))[::-1]
    width = heads * (2 * dim + 2 * vdim)
    proj = torch.randn(tokens, width + 8, generator=g).to(dtype).cuda()
    offsets = (0, heads * dim, 2 * heads * dim, 2 * heads * dim + heads * vdim)
    decay = torch.linspace(0.9, 0.99, heads).cuda()
    state = torch.randn(len(lengths), heads, dim, vdim, generator=g).cuda()
    old = state.cpu().double()
    weight = torch.rand(heads * vdim, generator=g).cuda() + 0.5
    starts = [sum(lengths[:i]) for i in range(len(lengths) + 1)]
    meta = lambda values: torch.tensor(values, dtype=torch.int32).cuda()
    positions = meta([t for n in lengths for t in range(n)])
    out = ops.retention(proj, offsets, None, None, 0, decay, state, meta(slots), positions, meta(starts), len(lengths),
                        heads, dim, vdim, 1e-6, dim ** -0.5, max(lengths), norm_span=span, norm_weight=weight, gate="sigmoid")
    p = proj.cpu().double()
    q, k = (p[:, o: o + heads * dim].view(tokens, heads, dim) for o in offsets[:2])
    v, gate = (p[:, o: o + heads * vdim].view(tokens, heads, vdim) for o in offsets[2:])
    f = decay.cpu().double()[:, None, None]
    for i, n in enumerate(lengths):
        S, size = old[slots[i]].clone(), old[slots[i]].abs()
        for t in range(starts[i], starts[i] + n):
            add = (k[t] * dim ** -0.5)[:, :, None] * v[t][:, None, :]
            S, size = f * S + add, f * size + add.abs()
            o, o_size = (S * q[t][:, :, None]).sum(1), (size * q[t].abs()[:, :, None]).sum(1)
            rms = torch.sqrt((o.view(heads // span, -1) ** 2).mean(-1) + 1e-6).repeat_interleave(span)[:, None]
            factor = weight.cpu().double().view(heads, vdim) * torch.sigmoid(gate[t]) / rms
            want = o * factor
            # float32 sums of n + dim terms and the powers of the decay in front of them, then the norm's own few roundings
            # (its sum of squares carries the error of all its columns)
            bound = (2 * n + dim + 16) * 2.0 ** -24 * (o_size + o_size.max() * want.abs() / factor.abs().clamp_min(1e-30) / rms) * factor.abs()
            if dtype == torch.bfloat16:
                bound = bound + 2.0 ** -8 * want.abs()
            assert torch.all((out[t].cpu().double().view(heads, vdim) - want).abs() <= bound + 1e-6)
        assert torch.all((state[slots[i]].cpu().double() - S).abs() <= (2 * n + 16) * 2.0 ** -24 * (size + 1))


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("lengths,heads,dim,vdim,rot,activation", [
    ((1,), 1, 1, 4, 0, None), ((1, 1, 1), 3, 9, 72, 4, "silu"), ((1,) * 5, 8, 128, 256, 128, None), ((1, 1), 2, 1024, 32, 0, None),
    ((1,), 2, 8, 1024, 6, "silu"), ((0, 2, 1, 1), 2, 72, 12, 72, None), ((1,) * 40, 4, 64, 64, 64, None)])
def test_retention_of_one_token_a_sequence(dtype, lengths, heads, dim, vdim, rot, activation):
    """The kernel that does a step in one workgroup a head, at the smallest and largest heads it takes, rows and columns
    that leave threads over, whole, partial and no rotation, and a sequence without a token beside one with two; against
    64 bits.  Columns that are no multiple of four, and a memory off a 16-byte line, take the general path."""
    from cie_amd.kernels import ops

    g = torch.Generator().manual_seed(6)
    tokens, slots = sum(lengths), list(range(len(lengths)))[::-1]
    assert ops.steps_retention(tokens, len(lengths), dim, vdim, 1)
    assert not ops.steps_retention(tokens, len(lengths), dim, vdim + 2, 1)
    assert not ops.steps_retention(tokens + 1, len(lengths), dim, vdim, 1)
    assert not ops.steps_retention(tokens, len(lengths), dim, vdim, 2)
    proj = torch.randn(tokens, heads * (2 * dim + 2 * vdim) + 3, generator=g).to(dtype).cuda()  # (rows off 16-byte lines)
    offsets = (3, 3 + heads * dim, 3 + 2 * heads * dim, 3 + 2 * heads * dim + heads * vdim)
    decay, weight = torch.linspace(0.9, 0.99, heads).cuda(), torch.rand(heads * vdim, generator=g).cuda() + 0.5
    kept = torch.randn(len(lengths), heads, dim, vdim, generator=g)
    starts = [sum(lengths[:i]) for i in range(len(lengths) + 1)]
    meta = lambda values: torch.tensor(values, dtype=torch.int32).cuda()
    at = torch.randint(0, 500, (tokens,), generator=g)
    angles = torch.arange(500)[:, None] * 0.7 ** torch.arange(rot // 2)[None, :]
    cos, sin = angles.cos().float().cuda(), angles.sin().float().cuda()
    run = lambda state: ops.retention(proj, offsets, cos if rot else None, sin if rot else None, rot, decay, state, meta(slots),
                                      meta(at.tolist()), meta(starts), len(lengths), heads, dim, vdim, 1e-6, 0.25, 499,
                                      activation=activation, norm_weight=weight)
    state = kept.cuda()
    off_line = torch.empty(kept.numel() + 1, device="cuda")[1:].view(kept.shape).copy_(kept)  # the general path
    out, general = run(state), run(off_line)
    p = proj.cpu().double()
    act = (lambda z: z * torch.sigmoid(z)) if activation else (lambda z: z)
    q, k = (act(p[:, o: o + heads * dim]).view(tokens, heads, dim) for o in offsets[:2])
    v, gate = (p[:, o: o + heads * vdim].view(tokens, heads, vdim) for o in offsets[2:])
    v = act(v)
    c, s = cos.cpu().double()[at][:, None], sin.cpu().double()[at][:, None]

    def turned(z):
        a, b, rest = z[..., :rot // 2], z[..., rot // 2: rot], z[..., rot:]
        size = torch.cat((a.abs() + b.abs(), a.abs() + b.abs(), rest.abs()), -1)
        return torch.cat((a * c - b * s, b * c + a * s, rest), -1), size

    (q, q_size), (k, k_size) = turned(q), turned(k)
    f = decay.cpu().double()[:, None, None]
    w = weight.cpu().double().view(heads, vdim)
    for i, n in enumerate(lengths):
        S, size = kept[slots[i]].double(), kept[slots[i]].double().abs()
        for t in range(starts[i], starts[i] + n):
            S = f * S + 0.25 * k[t][:, :, None] * v[t][:, None, :]
            size = f * size + 0.25 * k_size[t][:, :, None] * v[t].abs()[:, None, :]
            o, o_size = (S * q[t][:, :, None]).sum(1), (size * q_size[t][:, :, None]).sum(1)
            rms = torch.sqrt((o ** 2).mean(-1) + 1e-6)[:, None]
            factor = w * gate[t] * torch.sigmoid(gate[t]) / rms
            want = o * factor
            # a token's products, turns and activations are a dozen roundings each, o a float32 sum of dim terms, and the
            # root mean square carries the error of its columns (o_size.max() over |o|, in parts of rms)
            bound = (dim + 40) * 2.0 ** -24 * (o_size + o_size.max() * o.abs() / rms) * factor.abs()
            if dtype == torch.bfloat16:
                bound = bound + 2.0 ** -8 * want.abs()
            for result in (out, general):
                assert torch.all((result[t].cpu().double().view(heads, vdim) - want).abs() <= bound + 1e-6)
        for memory in (state, off_line):
            assert torch.all((memory[slots[i]].cpu().double() - S).abs() <= 40 * 2.0 ** -24 * (size + 1))


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("tokens,heads,plain,turned,latent,width,page_size", [
    (1, 16, 24, 32, 96, 128, 16), (7, 3, 5, 6, 11, 32, 4), (3, 40, 128, 64, 64, 256, 16), (300, 4, 16, 32, 96, 128, 32),
    (5, 2, 8, 0, 64, 64, 3), (2, 1, 1, 2, 1, 4, 1)])
@pytest.mark.parametrize("mode", ["turned", "unturned", "reads"])
def test_rows_and_entries_of_compressed_keys(dtype, tokens, heads, plain, turned, latent, width, page_size, mode):
    """Query rows and cache entries of one launch: heads that leave lanes over or take several workgroups, entries with and
    without zeros behind the latent, a part that does not turn or is not there, odd pages, a token without a page, and a
    layer that only reads; places that are nobody's stay as they are."""
    from cie_amd.kernels import ops

    if not turned and mode == "turned":
        mode = "unturned"
    g = torch.Generator().manual_seed(8)
    columns = heads * (plain + turned) + latent + turned
    proj = torch.randn(tokens, columns + 5, generator=g).to(dtype).cuda()[:, :columns]
    weight = torch.rand(latent, generator=g).cuda() + 0.5
    at = torch.randint(0, 40, (tokens,), generator=g)
    pages_each = -(-40 // page_size)
    table = torch.randperm(tokens * pages_each, generator=g).view(tokens, pages_each).int()
    lost = tokens - 1 if tokens > 2 else -1
    if lost >= 0:
        table[0, at[lost] // page_size] = -1  # (the last token's sequence has slot 0)
    slots = torch.arange(tokens).flip(0)
    angles = torch.arange(40)[:, None] * 0.7 ** torch.arange(turned // 2)[None, :]
    cos, sin = angles.cos().float(), angles.sin().float()
    keys = torch.full((tokens * pages_each, 1, page_size, width), 3.0, dtype=dtype, device="cuda")
    values = torch.full((tokens * pages_each, 1, width, page_size), 3.0, dtype=dtype, device="cuda")
    rows = ops.latent_rows(proj, weight, heads, plain, turned, latent, width, 1e-6,
                           (cos.cuda(), sin.cuda()) if mode == "turned" else None, at.int().cuda(),
                           torch.arange(tokens).int().cuda(), slots.int().cuda(), table.cuda(), keys, values,
                           write_kv=mode != "reads")
    p, c, s = proj.cpu().double(), cos.double()[at], sin.double()[at]
    half = turned // 2

    def turn(z):  # [tokens, ..., turned] -> turned, and what its roundings are relative to
        if mode != "turned":
            return z, z.abs()
        shape = (tokens,) + (1,) * (z.dim() - 2) + (half,)
        a, b, cc, ss = z[..., :half], z[..., half:], c.view(shape), s.view(shape)
        return torch.cat((a * cc - b * ss, b * cc + a * ss), -1), torch.cat((a.abs() + b.abs(),) * 2, -1)

    one = 2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -24  # the last rounding; four more of float32 in front of it
    close = lambda got, want, size: bool(((got.cpu().double() - want).abs() <= one * want.abs() + 4 * 2.0 ** -24 * size).all())
    q = rows.view(tokens, heads, width)
    want, size = turn(p[:, : heads * (plain + turned)].view(tokens, heads, plain + turned)[..., plain:])
    assert close(q[..., :turned], want, size) and not q[..., turned + latent:].any()
    down = p[:, heads * (plain + turned):]
    normed = down[:, :latent] / torch.sqrt((down[:, :latent] ** 2).mean(-1, keepdim=True) + 1e-6) * weight.cpu().double()
    key, key_size = turn(down[:, latent:])
    untouched = torch.ones(keys.shape[0], page_size, dtype=torch.bool)
    for t in range(tokens):
        page, row = int(table[slots[t], at[t] // page_size]), int(at[t] % page_size)
        if mode == "reads" or page < 0:
            continue
        untouched[page, row] = False
        k, v = keys[page, 0, row], values[page, 0, :, row]
        assert close(k[:turned], key[t], key_size[t]) and not v[:turned].any()
        for entry in (k, v):  # (the mean square: `latent` squares and their sum, a root, a quotient, two products)
            assert close(entry[turned: turned + latent], normed[t], (latent + 4) * normed[t].abs())
            assert not entry[turned + latent:].any()
    assert (keys.cpu()[:, 0][untouched] == 3).all() and (values.cpu()[:, 0].transpose(1, 2)[untouched] == 3).all()


@pytest.mark.parametrize("lengths,blocks,width,taps", [
    ((1,), 1, 8, 1), ((1,) * 5, 3, 24, 2), ((1,) * 16, 8, 256, 4), ((1,) * 17, 2, 264, 5), ((1, 0, 1, 0, 0), 2, 40, 4),
    ((1,) * 64, 4, 128, 4), ((1, 1), 1, 520, 3)])
def test_gated_recurrence_of_single_tokens(lengths, blocks, width, taps):
    """The kernel that makes the gates and moves the states, at blocks that end inside a tile of 16 channels, inside a slice
    of 32 and behind eight slices, rows that end inside a tile of 16 sequences, and places without a token, against the
    product and the walk by themselves."""
    from cie_amd.kernels import ops

    g = torch.Generator().manual_seed(9)
    tokens, channels = sum(lengths), blocks * width
    slots = list(range(len(lengths) + 2))[::-1][: len(lengths)]
    make = lambda *shape: torch.randn(*shape, generator=g)
    proj = make(tokens, 2 * channels + 1).bfloat16().cuda()  # (rows off 16-byte lines)
    y_pre, x_in = proj[:, 1: channels + 1], proj[:, channels + 1:]
    u = make(tokens, channels).bfloat16().cuda()
    weight, bias = (make(blocks, 2 * width, width) * width ** -0.5).bfloat16().cuda(), make(blocks, 2 * width).bfloat16().cuda()
    rate = -8.0 * torch.rand(channels, generator=g).cuda()
    state, past = make(len(lengths) + 2, channels).cuda(), make(len(lengths) + 2, max(taps - 1, 1), channels).cuda()
    state2, past2 = state.clone(), past.clone()
    starts = [sum(lengths[:i]) for i in range(len(lengths) + 1)]
    meta = lambda values: torch.tensor(values, dtype=torch.int32).cuda()
    takes, n = ops.steps_gated_recurrence, len(lengths)
    assert takes(u, weight, n, width, taps) and not takes(u.float(), weight, n, width, taps)
    assert not takes(u, weight, n, width + 4, taps) and not takes(u, weight, n, width, 6)
    assert not takes(u, weight, 16 * 5 * 256 + 1, width, taps)
    out = ops.gated_recurrence_step(y_pre, x_in, u, weight, bias, rate, state, past, meta(slots), meta(starts), len(lengths), taps)
    gates = ops.block_linear(u, weight, bias, out_dtype=torch.float32)
    want = ops.gated_recurrence(y_pre, x_in, u, gates, width, rate, state2, past2, meta(slots), meta(starts), len(lengths), taps)
    # float32 sums of `width` terms of some 1 / sqrt(width) in another order, through slopes of at most 2 (the
    # decay's, |rate| / 4) and the state's size of some 4; the bfloat16 result is rounded once, either way
    near = width * 2.0 ** -24 * 8 + 1e-6
    assert torch.allclose(state, state2, atol=near, rtol=near)
    assert torch.allclose(out.float(), want.float(), atol=4 * near, rtol=2.0 ** -7)
    assert torch.equal(past, past2)


@pytest.mark.parametrize("lengths,blocks,width,taps", [
    ((2,), 1, 64, 1), ((64, 1, 129), 3, 64, 4), ((63, 65, 1, 1, 2), 8, 128, 4), ((1, 700), 2, 256, 3), ((17,) * 9, 1, 256, 4),
    ((1999,), 8, 256, 4), ((3, 0, 61, 0, 1), 5, 128, 2)])
def test_gated_recurrence_in_chunks(lengths, blocks, width, taps):
    """Sequences that begin, end or both inside a chunk, at its first and last token, one over many chunks, and places without
    a token, against the product and the walk by themselves; a sequence whose state is infinite keeps that to itself."""
    from cie_amd.kernels import ops

    g = torch.Generator().manual_seed(10)
    tokens, channels = sum(lengths), blocks * width
    slots = list(range(len(lengths) + 2))[::-1][: len(lengths)]
    make = lambda *shape: torch.randn(*shape, generator=g)
    proj = make(tokens, 2 * channels + 8).bfloat16().cuda()
    y_pre, x_in = proj[:, 8: channels + 8], proj[:, channels + 8:]
    u = make(tokens, channels).bfloat16().cuda()
    weight, bias = (make(blocks, 2 * width, width) * width ** -0.5).bfloat16().cuda(), make(blocks, 2 * width).bfloat16().cuda()
    rate = -8.0 * torch.rand(channels, generator=g).cuda()
    state, past = make(len(lengths) + 2, channels).cuda(), make(len(lengths) + 2, max(taps - 1, 1), channels).cuda()
    starts = [sum(lengths[:i]) for i in range(len(lengths) + 1)]
    meta = lambda values: torch.tensor(values, dtype=torch.int32).cuda()
    of_token = meta([i for i, n in enumerate(lengths) for _ in range(n)])
    assert ops.chunks_gated_recurrence(y_pre, u, weight, width, taps)
    assert not ops.chunks_gated_recurrence(proj[:, 1: channels + 1], u, weight, width, taps)
    assert not ops.chunks_gated_recurrence(y_pre, u.float(), weight, width, taps)
    assert not ops.chunks_gated_recurrence(y_pre, u, weight, 32, taps)
    for odd in (None, math.inf, math.nan):
        if odd is not None:
            state[slots[0], 3::7] = odd
        state2, past2 = state.clone(), past.clone()
        out = ops.gated_recurrence_chunks(y_pre, x_in, u, weight, bias, rate, state, past, of_token, meta(slots), meta(starts),
                                          len(lengths), taps)
        gates = ops.block_linear(u, weight, bias, out_dtype=torch.float32)
        want = ops.gated_recurrence(y_pre, x_in, u, gates, width, rate, state2, past2, meta(slots), meta(starts), len(lengths), taps)
        # as above; what fades joins in another order (a product of fades is some log2(64) + 4 roundings off)
        near = width * 2.0 ** -24 * 8 + 2e-6
        there = torch.isfinite(state2)
        assert torch.allclose(state[there], state2[there], atol=near, rtol=near)
        assert torch.equal(torch.isfinite(out[lengths[0]:]), torch.isfinite(want[lengths[0]:]))
        there = torch.isfinite(want)
        assert torch.allclose(out[there].float(), want[there].float(), atol=4 * near, rtol=2.0 ** -7)
        assert torch.equal(past, past2)


def test_gated_recurrence_in_chunks_is_as_near_to_64_bits_as_the_walk():
    """The states of a portion in chunks, whose tokens compose by doubling, and those of the walk in order, at the fades of a model
    whose parameters are drawn about zero."""
    from cie_amd.kernels import ops

    blocks, width, taps, off = 2, 256, 4, {"chunks": 0.0, "walk": 0.0}
    channels = blocks * width
    meta = lambda values: torch.tensor(values, dtype=torch.int32).cuda()  # noqa: E731
    for seed, lengths in enumerate([(61, 128, 97, 33, 80, 111, 20, 49), (300, 17, 449), (640,), (255, 257)]):
        g = torch.Generator().manual_seed(30 + seed)
        make = lambda *shape: torch.randn(*shape, generator=g)  # noqa: E731, B023
        tokens, n = sum(lengths), len(lengths)
        proj, u = make(tokens, 2 * channels).bfloat16().cuda(), make(tokens, channels).bfloat16().cuda()
        weight, bias = (make(blocks, 2 * width, width) * width ** -0.5).bfloat16().cuda(), make(blocks, 2 * width).bfloat16().cuda()
        rate = -8.0 * torch.nn.functional.softplus(0.02 * make(channels)).cuda()
        state, past = make(n, channels).cuda(), make(n, taps - 1, channels).cuda()
        starts = [sum(lengths[:i]) for i in range(n + 1)]
        rows = u.double().view(tokens, blocks, width).transpose(0, 1)
        gates = torch.matmul(rows, weight.double().transpose(1, 2).contiguous()) + bias.double()[:, None]
        gates = gates.transpose(0, 1).reshape(tokens, blocks, 2, width)
        log_fade = rate.double() * torch.sigmoid(gates[:, :, 0]).reshape(tokens, channels)
        fade, add = torch.exp(log_fade), torch.sqrt(-torch.expm1(2 * log_fade)) * torch.sigmoid(gates[:, :, 1]).reshape(tokens, channels) * u.double()
        want = state.double()
        for i in range(n):
            for t in range(starts[i], starts[i + 1]):
                want[i] = torch.addcmul(add[t], fade[t], want[i])
        for name in off:
            mine, kept = state.clone(), past.clone()
            if name == "chunks":
                ops.gated_recurrence_chunks(proj[:, :channels], proj[:, channels:], u, weight, bias, rate, mine, kept,
                                            meta([i for i, k in enumerate(lengths) for _ in range(k)]), meta(range(n)), meta(starts), n, taps)
            else:
                ops.gated_recurrence(proj[:, :channels], proj[:, channels:], u, ops.block_linear(u, weight, bias, out_dtype=torch.float32),
                                     width, rate, mine, kept, meta(range(n)), meta(starts), n, taps)
            off[name] += float(((mine.double() - want).norm() / want.norm()) ** 2)
    # (a token has the walk's own rounding and what fades of those in front, which is the same or, at a chunk's first tokens, one more)
    assert off["chunks"] ** 0.5 <= 1.05 * off["walk"] ** 0.5, off


def test_gated_recurrence_in_chunks_of_very_many_sequences():
    """More sequences and groups of tokens together than a grid's second dimension holds, as the product and the walk take them."""
    from cie_amd.kernels import ops

    lengths, width, taps = (1,) * 64990 + (20000,), 64, 2
    g = torch.Generator().manual_seed(11)
    tokens, n = sum(lengths), len(lengths)
    proj, u = (torch.randn(tokens, k * width, generator=g).bfloat16().cuda() for k in (2, 1))
    weight, bias = (torch.randn(1, 2 * width, width, generator=g) * width ** -0.5).bfloat16().cuda(), torch.zeros(1, 2 * width).bfloat16().cuda()
    rate = -8.0 * torch.rand(width, generator=g).cuda()
    state, past = torch.randn(n, width, generator=g).cuda(), torch.randn(n, 1, width, generator=g).cuda()
    of_token, slots = torch.arange(tokens, dtype=torch.int32).clamp(max=n - 1).cuda(), torch.arange(n, dtype=torch.int32).cuda()
    starts = torch.tensor([*range(n), tokens], dtype=torch.int32).cuda()
    state2, past2 = state.clone(), past.clone()
    out = ops.gated_recurrence_chunks(proj[:, :width], proj[:, width:], u, weight, bias, rate, state, past, of_token, slots, starts, n, taps)
    want = ops.gated_recurrence(proj[:, :width], proj[:, width:], u, ops.block_linear(u, weight, bias, out_dtype=torch.float32), width, rate,
                                state2, past2, slots, starts, n, taps)
    near = width * 2.0 ** -24 * 8 + 2e-6  # (as above)
    assert torch.allclose(state, state2, atol=near, rtol=near) and torch.equal(past, past2)
    assert torch.allclose(out.float(), want.float(), atol=4 * near, rtol=2.0 ** -7)


@pytest.mark.parametrize("joined", [True, False])
@pytest.mark.parametrize("name", sorted(pu.SMALL))
def test_layers_whose_first_products_run_in_one_launch(models, name, joined, monkeypatch):
    """Single tokens through layers whose branches start in one launch and end in one, or, where the last products' columns are too
    many for that, in one each; against the plain implementation."""
    from cie_amd.parts import block, linear

    raw, weights, requests, plain = models[name]
    if not joined:
        monkeypatch.setattr(linear, "PART_BELOW_TILES", 1)
    begun, ended = [], []
    for kept, which in ((begun, "silu_beside"), (ended, "parts_beside")):
        monkeypatch.setattr(block, which, lambda *a, kept=kept, real=getattr(block, which): (kept.append(real(*a)), kept[-1])[1])
    run_and_compare(raw, weights, requests, replay_util.tail_one_by_one(requests, tail=8), "bfloat16", plain)
    assert any(out is not None for out in begun) and ended and all((out is not None) == joined for out in ended)
