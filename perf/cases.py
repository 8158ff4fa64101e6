"""The work that a program serving an int8 Qwen3 with this package has it do, as timed cases.

Every case goes through the package's public entry points: ``Int8Linear.forward``,
``Qwen3ForCausalLM.forward`` / ``ModelRunner.prepare`` / ``forward_logits``, ``paged_attention`` and
``sample``. Two model shapes are used, those of ``workloads.QWEN3_0_6B`` and ``workloads.QWEN3_8B``,
with seeded random weights quantized to int8. A kind of work is one of:

  linear     one ``Int8Linear.forward`` call, as a program with its own layers makes it
  decode     one token for each of a batch of running sequences, through a slice of decoder layers
             captured as a HIP graph (decode steps are replayed from graphs when a model is served)
  prompts    prompt chunks (with or without cached tokens before them) through a slice of decoder
             layers, launched eagerly with the batch's plan built on the host, as prefill steps are
  step       the whole model to the logits of the sampled rows: a captured decode step, or an eager
             mixed step of running sequences with one prompt chunk
  attention  one layer's ``paged_attention`` call: cache write and attention through block tables
  sample     next tokens from logits with each request's own settings

Lengths are spread evenly over [lo, hi] in a fixed, unsorted order, so that the work of a case is
known from the case alone; weights, activations, caches, block tables and tokens come from the seed.
"""

from __future__ import annotations

import math
from dataclasses import dataclass
from typing import Any

import torch

from miniserve_amd import workloads
from miniserve_amd.attention.backends import SeqChunk, build_attention_metadata, paged_attention
from miniserve_amd.model.qwen3 import Qwen3Config
from miniserve_amd.quant.int8 import Int8Linear, quantize_int8_
from miniserve_amd.runner.model_runner import ModelRunner, ScheduledChunk
from miniserve_amd.runner.sampler import sample

ARCH = {"0.6b": workloads.QWEN3_0_6B, "8b": workloads.QWEN3_8B}
BLOCK = 16
SLICE_VOCAB = 8192  # a slice of layers looks its tokens up in a small embedding
PROJECTIONS = {  # (out, in) features of the two models' linears
    "0.6b": {"qkv": (4096, 1024), "o": (1024, 2048), "gate": (3072, 1024), "gate_up": (6144, 1024), "down": (1024, 3072)},
    "8b": {"qkv": (6144, 4096), "o": (4096, 4096), "gate": (12288, 4096), "gate_up": (24576, 4096), "down": (4096, 12288)},
}


# ---- the cases ------------------------------------------------------------------------------------


def listed() -> list[dict[str, Any]]:
    return [
        # A single projection for a small batch: launch and latency.
        {"name": "linear-16", "kind": "linear", "out": 3072, "in": 1024, "tokens": 16},
        # One user's chat with the 8B shape: nothing to batch, all weights read for one token.
        {"name": "decode-8b-1", "kind": "decode", "arch": "8b", "layers": 2, "batch": 1, "lo": 1100, "hi": 1100},
        # A small server of the 8B shape: an odd batch at chat lengths.
        {"name": "decode-8b-27", "kind": "decode", "arch": "8b", "layers": 2, "batch": 27, "lo": 200, "hi": 2000},
        # A full server of the 8B shape: the keys and values are most of the bytes.
        {"name": "decode-8b-256", "kind": "decode", "arch": "8b", "layers": 2, "batch": 256, "lo": 512, "hi": 4096},
        # The small model's whole decode step at the batch its benchmark runs.
        {"name": "step-0.6b-64", "kind": "step", "arch": "0.6b", "layers": 28, "batch": 64, "lo": 256, "hi": 384, "chunk": 0},
        # Its mixed step: 64 running sequences and a long prompt's chunk.
        {"name": "step-0.6b-mixed", "kind": "step", "arch": "0.6b", "layers": 28, "batch": 64, "lo": 64, "hi": 1024, "chunk": 1984},
        # A handful of short chat prompts arriving together: ragged, a few hundred tokens.
        {"name": "prompts-8b-short", "kind": "prompts", "arch": "8b", "layers": 2, "batch": 5, "lo": 40, "hi": 260, "cached": 0},
        # Long fresh prompts: the matrix products are most of the work.
        {"name": "prompts-8b-long", "kind": "prompts", "arch": "8b", "layers": 2, "batch": 2, "lo": 2048, "hi": 2048, "cached": 0},
        # Attention of a running batch at mixed lengths.
        {"name": "attn-decode-64", "kind": "attention", "heads": 16, "kv_heads": 8, "batch": 64, "new": 1, "lo": 128, "hi": 2048},
        # A few sequences with very long contexts: the batch alone does not fill the chip.
        {"name": "attn-decode-long", "kind": "attention", "heads": 32, "kv_heads": 8, "batch": 3, "new": 1, "lo": 20000, "hi": 32768},
        # A later chunk of a long document: many new tokens after many cached ones.
        {"name": "attn-chunk-cached", "kind": "attention", "heads": 32, "kv_heads": 8, "batch": 1, "new": 2000, "lo": 8000, "hi": 8000},
        # Next tokens of a batch whose requests have settings of their own.
        {"name": "sample-64", "kind": "sample", "rows": 64, "vocab": 151936, "settings": "mixed"},
    ]


def _log(rng: Any, lo: int, hi: int) -> int:
    """A whole number between lo and hi, spread over its logarithm."""
    return max(lo, min(hi, round(math.exp(rng.uniform(math.log(lo), math.log(hi))))))


def draw(rng: Any) -> dict[str, Any]:
    kind = rng.choice(["linear", "decode", "decode", "prompts", "prompts", "step", "attention", "attention", "sample"])
    arch = rng.choice(["0.6b", "8b"])
    if kind == "linear":
        out, inner = PROJECTIONS[arch][rng.choice(sorted(PROJECTIONS[arch]))]
        return {"kind": kind, "out": out, "in": inner, "tokens": _log(rng, 1, 4096)}
    if kind == "decode":
        lo = _log(rng, 32, 2048)
        return {"kind": kind, "arch": arch, "layers": 2, "batch": _log(rng, 1, 256), "lo": lo, "hi": min(4096, lo + _log(rng, 16, 3000))}
    if kind == "prompts":
        total = _log(rng, 130, 4096)
        batch = rng.randint(1, max(1, min(8, total // 40)))
        mid = total // batch
        spread = rng.randint(0, mid // 2)
        return {"kind": kind, "arch": arch, "layers": 2, "batch": batch, "lo": mid - spread, "hi": mid + spread,
                "cached": rng.choice([0, 0, rng.randint(1, 2048)])}
    if kind == "step":
        lo = _log(rng, 32, 512)
        chunk = rng.choice([0, _log(rng, 130, 1984)])
        return {"kind": kind, "arch": "0.6b", "layers": 28, "batch": _log(rng, 1, 128) if not chunk else _log(rng, 1, 64),
                "lo": lo, "hi": lo + _log(rng, 16, 512), "chunk": chunk}
    if kind == "attention":
        heads = {"0.6b": 16, "8b": 32}[arch]
        what = rng.choice(["decode", "long", "chunk", "verify"])
        if what == "decode":
            lo = _log(rng, 32, 2048)
            return {"kind": kind, "heads": heads, "kv_heads": 8, "batch": _log(rng, 8, 256), "new": 1, "lo": lo, "hi": lo + _log(rng, 16, 2048)}
        if what == "long":
            lo = _log(rng, 4096, 24000)
            return {"kind": kind, "heads": heads, "kv_heads": 8, "batch": rng.randint(1, 6), "new": 1, "lo": lo, "hi": lo + rng.randint(0, 8000)}
        if what == "verify":
            lo = _log(rng, 64, 2048)
            return {"kind": kind, "heads": heads, "kv_heads": 8, "batch": _log(rng, 4, 64), "new": rng.randint(2, 8), "lo": lo, "hi": lo + _log(rng, 16, 1024)}
        new = _log(rng, 130, 2048)
        lo = new + rng.choice([0, _log(rng, 16, 6000)])
        return {"kind": kind, "heads": heads, "kv_heads": 8, "batch": 1, "new": new, "lo": lo, "hi": lo}
    return {"kind": kind, "rows": _log(rng, 1, 96), "vocab": 151936, "settings": rng.choice(["mixed", "top_k", "top_p", "temperature"])}


# ---- shapes that follow from a case -----------------------------------------------------------------


def _spread(n: int, lo: int, hi: int) -> list[int]:
    """n lengths in [lo, hi], evenly spread, in an order that is neither rising nor falling."""
    return [lo + int((hi - lo) * ((0.5 + 0.6180339887498949 * i) % 1.0)) for i in range(n)]


def _chunks(case: dict[str, Any]) -> list[tuple[int, int]]:
    """(cached tokens, new tokens) of every sequence of a case."""
    lengths = _spread(case["batch"], case["lo"], case["hi"])
    if case["kind"] == "prompts":
        return [(case["cached"], n) for n in lengths]
    if case["kind"] == "attention":
        return [(c - case["new"], case["new"]) for c in lengths]
    return [(c - 1, 1) for c in lengths] + ([(0, case["chunk"])] if case.get("chunk") else [])


def _config(case: dict[str, Any]) -> dict[str, Any]:
    cfg = {**ARCH[case["arch"]], "num_hidden_layers": case["layers"]}
    if case["kind"] != "step":
        cfg.update(vocab_size=SLICE_VOCAB, tie_word_embeddings=True)  # the slice ends before the LM head
    return cfg


def _positions(chunks: list[tuple[int, int]]) -> int:
    return -(-max(c + n for c, n in chunks) // 256) * 256


def _attended(chunks: list[tuple[int, int]]) -> int:
    """(query, key) pairs under the causal mask."""
    return sum(n * c + n * (n + 1) // 2 for c, n in chunks)


def work(case: dict[str, Any]) -> dict[str, float]:
    kind = case["kind"]
    if kind == "linear":
        m, n, k = case["tokens"], case["out"], case["in"]
        return {"bytes": n * k + 2 * n + 2 * m * (n + k), "flops": 2.0 * m * n * k}
    if kind == "sample":
        return {"bytes": 4.0 * case["rows"] * case["vocab"] + 8 * case["rows"], "flops": 0.0}
    chunks = _chunks(case)
    tokens, keys = sum(n for _, n in chunks), sum(c + n for c, n in chunks)
    if kind == "attention":
        h, kvh, d = case["heads"], case["kv_heads"], 128
        return {"bytes": 4.0 * kvh * d * keys + 4.0 * tokens * h * d + 8.0 * tokens * kvh * d, "flops": 4.0 * h * d * _attended(chunks)}
    cfg = _config(case)
    hid, inter, d = cfg["hidden_size"], cfg["intermediate_size"], cfg["head_dim"]
    h, kvh = cfg["num_attention_heads"], cfg["num_key_value_heads"]
    rows = (h + 2 * kvh) * d + hid + 2 * inter + hid
    params = (h + 2 * kvh) * d * hid + h * d * hid + 3 * hid * inter
    layer_bytes = params + 2 * rows + 4.0 * kvh * d * keys  # int8 weights, scales, keys and values (the new ones written)
    layer_flops = 2.0 * tokens * params + 4.0 * h * d * _attended(chunks)
    nbytes, flops = layer_bytes * cfg["num_hidden_layers"], layer_flops * cfg["num_hidden_layers"]
    if kind == "step":
        sampled = len(chunks)
        nbytes += 2.0 * cfg["vocab_size"] * hid + 4.0 * sampled * cfg["vocab_size"]
        flops += 2.0 * sampled * cfg["vocab_size"] * hid
    else:
        nbytes += 4.0 * tokens * hid  # embedding rows in, hidden states out
    return {"bytes": nbytes, "flops": flops}


def tolerance(case: dict[str, Any]) -> Any:
    kind = case["kind"]
    if kind == "sample":
        # Token ids: equal but for a race whose best two scores are within float32 rounding.
        return {"rel": 0.0, "differ": 0.01}
    if kind == "linear":
        return {"rel": 0.007, "max": 0.05}  # one bf16 rounding of the result; 1.7e-3 from 64 bits
    if kind == "attention":
        return {"rel": 0.01, "max": 0.1}
    return {"rel": 0.03, "max": 0.5}


# ---- inputs -----------------------------------------------------------------------------------------


@dataclass(frozen=True)
class Params:
    """A request's sampling settings, as an engine hands them to the sampler."""

    temperature: float
    top_k: int
    top_p: float
    greedy: bool


SETTINGS = {
    "temperature": [Params(0.8, -1, 1.0, False)],
    "top_p": [Params(0.7, -1, 0.95, False)],
    "top_k": [Params(0.6, 20, 0.95, False), Params(1.0, 50, 1.0, False)],
    "mixed": [Params(0.7, -1, 0.95, False), Params(0.0, -1, 1.0, True), Params(0.6, 20, 0.95, False), Params(0.8, -1, 1.0, False)],
}


def _generator(seed: int) -> torch.Generator:
    return torch.Generator(device="cuda").manual_seed(seed)


def _tables(chunks: list[tuple[int, int]], seed: int) -> tuple[list[list[int]], int]:
    """Block tables over a pool that holds just these sequences, in a random order of blocks."""
    need = [-(-(c + n) // BLOCK) for c, n in chunks]
    perm = torch.randperm(sum(need), generator=torch.Generator().manual_seed(seed)).tolist()
    tables, off = [], 0
    for n in need:
        tables.append(perm[off : off + n])
        off += n
    return tables, sum(need)


def _slots(chunks: list[tuple[int, int]], tables: list[list[int]]) -> list[int]:
    return [t[p // BLOCK] * BLOCK + p % BLOCK for (c, n), t in zip(chunks, tables) for p in range(c, c + n)]


def _weights(case: dict[str, Any], seed: int) -> dict[str, torch.Tensor]:
    """Random weights; the whole model gets a wide embedding that keeps each token visible in the last
    hidden state, as training does: without it 28 layers of noise blow up every rounding (two of this
    package's own routes differ by 3e-2 in the logits at a spread of 0.4, by 1.3e-2 at 2.0)."""
    return workloads.random_weights(_config(case), seed, norm_jitter=0.1, device="cuda",
                                    embed_std=2.0 if case["kind"] == "step" else None)


def _scheduled(case: dict[str, Any], seed: int) -> tuple[list[ScheduledChunk], int]:
    chunks = _chunks(case)
    tables, blocks = _tables(chunks, seed)
    vocab = _config(case)["vocab_size"]
    g = torch.Generator().manual_seed(seed + 1)
    return [ScheduledChunk(torch.randint(0, vocab, (c + n,), generator=g).tolist(), c, n, t)
            for (c, n), t in zip(chunks, tables)], blocks


def _linear_inputs(case: dict[str, Any], seed: int) -> tuple[torch.Tensor, torch.Tensor]:
    g = _generator(seed)
    w = (torch.randn(case["out"], case["in"], generator=g, device="cuda") * 0.02).to(torch.bfloat16)
    return w, torch.randn(case["tokens"], case["in"], generator=g, device="cuda").to(torch.bfloat16)


def _attention_inputs(case: dict[str, Any], seed: int) -> dict[str, Any]:
    chunks = _chunks(case)
    tables, blocks = _tables(chunks, seed)
    g = _generator(seed)
    t, kvh = sum(n for _, n in chunks), case["kv_heads"]

    def normal(*shape: int) -> torch.Tensor:
        return torch.randn(*shape, generator=g, device="cuda").to(torch.bfloat16)

    return {"chunks": chunks, "tables": tables, "slots": _slots(chunks, tables), "q": normal(t, case["heads"], 128),
            "k": normal(t, kvh, 128), "v": normal(t, kvh, 128), "k_cache": normal(blocks * BLOCK, kvh, 128),
            "v_cache": normal(blocks * BLOCK, kvh, 128)}


def _logits(case: dict[str, Any], seed: int) -> torch.Tensor:
    """Logits as a language model has them: a broad bulk, a few likely tokens (some rows sure, others
    not), rounded to bf16 as the head's product is."""
    g = _generator(seed)
    r, v = case["rows"], case["vocab"]
    x = torch.randn(r, v, generator=g, device="cuda") * 2.0
    likely = torch.randint(0, v, (r, 40), generator=g, device="cuda")
    lift = torch.rand(r, 40, generator=g, device="cuda") * (6.0 + 12.0 * torch.rand(r, 1, generator=g, device="cuda"))
    return x.scatter_add_(1, likely, lift).to(torch.bfloat16).float()


def prepare(case: dict[str, Any], seed: int) -> dict[str, Any]:
    kind = case["kind"]
    if kind == "linear":
        w, x = _linear_inputs(case, seed)
        return {"kind": kind, "layer": Int8Linear(w), "x": x}
    if kind == "sample":
        options = SETTINGS[case["settings"]]
        return {"kind": kind, "logits": _logits(case, seed), "params": [options[i % len(options)] for i in range(case["rows"])], "seed": seed}
    if kind == "attention":
        s = _attention_inputs(case, seed)
        seqs, flat = [], 0
        for (c, n), t in zip(s["chunks"], s["tables"]):
            seqs.append(SeqChunk(flat, n, c, t))
            flat += n
        slots = torch.tensor(s["slots"], dtype=torch.int64, device="cuda")
        meta = build_attention_metadata(seqs, slots, BLOCK)
        return {"kind": kind, "args": (s["q"], s["k"], s["v"], s["k_cache"], s["v_cache"], meta, 128**-0.5)}
    device = torch.device("cuda", torch.cuda.current_device())
    positions = _positions(_chunks(case))
    model = workloads.build_model(_config(case), _weights(case, seed), device, positions)
    quantize_int8_(model)
    runner = ModelRunner(model, device, max_model_len=positions)
    scheduled, blocks = _scheduled(case, seed)
    runner.allocate_kv_cache(blocks)
    workloads.fill_kv_pool_(runner.kv_cache, seed + 2, on_device=True)
    state = {"kind": kind, "runner": runner, "scheduled": scheduled}
    if kind == "decode" or (kind == "step" and not case["chunk"]):
        _capture(state)
    return state


def _forward(state: dict[str, Any], inp: Any) -> torch.Tensor:
    runner = state["runner"]
    if state["kind"] == "step":
        return runner.forward_logits(inp)
    with torch.inference_mode():
        return runner.model(inp.input_ids, inp.positions, runner.kv_caches, inp.attn)


def _capture(state: dict[str, Any]) -> None:
    """The decode step as a graph with static inputs, the handle that a serving loop replays."""
    inp = state["runner"].prepare(state["scheduled"])
    stream = torch.cuda.Stream()
    stream.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(stream):
        for _ in range(2):
            _forward(state, inp)
    torch.cuda.current_stream().wait_stream(stream)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=stream):
        out = _forward(state, inp)
    state.update(graph=graph, inp=inp, out=out)


def run(state: dict[str, Any]) -> Any:
    kind = state["kind"]
    if kind == "linear":
        return state["layer"](state["x"])
    if kind == "attention":
        args = state["args"]
        return {"out": paged_attention(*args), "k_cache": args[3], "v_cache": args[4]}
    if kind == "sample":
        params = state["params"]
        torch.cuda.manual_seed(state["seed"])  # a reproducible server: the noise follows from the seed
        return sample(state["logits"], params, [None] * len(params))
    if "graph" in state:
        state["graph"].replay()
        out = state["out"]
    else:
        out = _forward(state, state["runner"].prepare(state["scheduled"]))
    return {"logits" if kind == "step" else "hidden": out, "kv": state["runner"].kv_cache}


# ---- the same in 64 bits ------------------------------------------------------------------------------


def _dequantized(w: torch.Tensor) -> torch.Tensor:
    """The weights an int8 linear multiplies with: bf16(q * s), s = bf16(max|row| / 127)."""
    s = w.float().abs().amax(dim=1).clamp(min=1e-8) / 127.0
    q = torch.round(w.float() / s[:, None]).clamp(-127, 127)
    return (q.to(torch.bfloat16) * s.to(torch.bfloat16)[:, None]).double()


def _attend(q: torch.Tensor, kc: torch.Tensor, vc: torch.Tensor, chunks: list[tuple[int, int]], tables: list[list[int]]) -> torch.Tensor:
    """Causal attention of every sequence's new tokens: q [T, H, D], caches [slots, KVH, D], float64."""
    out, flat = torch.empty_like(q), 0
    kvh, d = kc.shape[1], kc.shape[2]
    group = q.shape[1] // kvh
    for (c, n), table in zip(chunks, tables):
        pos = torch.arange(c + n, device=q.device)
        slots = torch.tensor(table, device=q.device)[pos // BLOCK] * BLOCK + pos % BLOCK
        k, v = kc[slots].permute(1, 2, 0).contiguous(), vc[slots].permute(1, 0, 2).contiguous()
        qs = q[flat : flat + n].view(n, kvh, group, d).permute(1, 2, 0, 3).reshape(kvh, group * n, d).contiguous()
        scores = torch.bmm(qs, k).mul_(d**-0.5).view(kvh, group, n, c + n)
        scores.masked_fill_(pos[None, :] > c + torch.arange(n, device=q.device)[:, None], float("-inf"))
        o = torch.bmm(scores.softmax(-1).view(kvh, group * n, c + n), v)
        out[flat : flat + n] = o.view(kvh, group, n, d).permute(2, 0, 1, 3).reshape(n, kvh * group, d)
        flat += n
    return out


def _norm(x: torch.Tensor, w: torch.Tensor, eps: float) -> torch.Tensor:
    return x * torch.rsqrt(x.pow(2).mean(-1, keepdim=True) + eps) * w.double()


def _rotated(x: torch.Tensor, cos: torch.Tensor, sin: torch.Tensor) -> torch.Tensor:
    a, b = x.chunk(2, dim=-1)
    return x * cos[:, None] + torch.cat([-b, a], dim=-1) * sin[:, None]


def _exact_model(case: dict[str, Any], seed: int) -> dict[str, torch.Tensor]:
    cfg, w = Qwen3Config.from_dict(_config(case)), _weights(case, seed)
    chunks = _chunks(case)
    scheduled, blocks = _scheduled(case, seed)
    tables = [s.block_table for s in scheduled]
    h, kvh, d, eps = cfg.num_attention_heads, cfg.num_key_value_heads, cfg.head_dim, cfg.rms_norm_eps
    kv = torch.zeros(cfg.num_hidden_layers, 2, blocks * BLOCK, kvh, d, dtype=torch.bfloat16, device="cuda")
    workloads.fill_kv_pool_(kv, seed + 2, on_device=True)
    kv = kv.double()
    ids = torch.tensor([t for s in scheduled for t in s.token_ids[s.num_computed : s.num_computed + s.num_new]], device="cuda")
    pos = torch.tensor([p for c, n in chunks for p in range(c, c + n)], device="cuda")
    slots = torch.tensor(_slots(chunks, tables), device="cuda")
    # The rotary tables are inputs: float32 angles, rounded to bf16 as the model's q and k are.
    inv = 1.0 / (cfg.rope_theta ** (torch.arange(0, d, 2, dtype=torch.int64).float() / d))
    angles = torch.arange(_positions(chunks), dtype=torch.float32)[:, None] * inv[None, :]
    angles = torch.cat([angles, angles], dim=-1)
    cos, sin = (f(angles).to(torch.bfloat16).double().cuda()[pos] for f in (torch.cos, torch.sin))
    x = w["embed_tokens.weight"][ids].double()
    for i in range(cfg.num_hidden_layers):
        p = f"layers.{i}."

        def linear(name: str, a: torch.Tensor) -> torch.Tensor:
            return a @ _dequantized(w[p + name + ".weight"]).t().contiguous()

        qkv = linear("self_attn.qkv_proj", _norm(x, w[p + "input_layernorm.weight"], eps))
        q, k, v = (t.view(t.shape[0], -1, d) for t in qkv.split([h * d, kvh * d, kvh * d], dim=-1))
        q = _rotated(_norm(q, w[p + "self_attn.q_norm.weight"], eps), cos, sin)
        kv[i, 0, slots] = _rotated(_norm(k, w[p + "self_attn.k_norm.weight"], eps), cos, sin)
        kv[i, 1, slots] = v
        x = x + linear("self_attn.o_proj", _attend(q, kv[i, 0], kv[i, 1], chunks, tables).reshape(len(ids), h * d))
        gate, up = linear("mlp.gate_up_proj", _norm(x, w[p + "post_attention_layernorm.weight"], eps)).chunk(2, dim=-1)
        x = x + linear("mlp.down_proj", torch.nn.functional.silu(gate) * up)
    x = _norm(x, w["norm.weight"], eps)
    if case["kind"] != "step":
        return {"hidden": x, "kv": kv}
    last = torch.tensor([n for _, n in chunks], device="cuda").cumsum(0) - 1
    head = w["embed_tokens.weight"] if cfg.tie_word_embeddings else w["lm_head.weight"]
    return {"logits": x[last] @ head.double().t().contiguous(), "kv": kv}


def exact(case: dict[str, Any], seed: int) -> Any:
    kind = case["kind"]
    if kind == "linear":
        w, x = _linear_inputs(case, seed)
        return x.double() @ _dequantized(w).t().contiguous()
    if kind == "sample":
        return None  # token ids: no value between two of them
    if kind == "attention":
        s = _attention_inputs(case, seed)
        kc, vc = s["k_cache"].double(), s["v_cache"].double()
        slots = torch.tensor(s["slots"], device="cuda")
        kc[slots], vc[slots] = s["k"].double(), s["v"].double()
        return {"out": _attend(s["q"].double(), kc, vc, s["chunks"], s["tables"]), "k_cache": kc, "v_cache": vc}
    return _exact_model(case, seed)
