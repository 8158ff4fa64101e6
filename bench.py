"""Throughput of MiniServe's int8 hot path on one MI355X.

    python bench.py [--gpus 1] [--steps K] [--warmup W] [--no-cpu-baseline] [--workload NAME]

Default workload ``decode`` -- the headline metric: decode tok/s of a Qwen3-0.6B-architecture
int8 model at batch 64. One step = what the runner does per engine step: build the flat batch and
attention metadata on the host, upload it (pinned, non-blocking), run the 28 layers, the final
norm + LM head + greedy argmax on the 64 sampled rows, and the one device->host sync; the step is
a captured HIP graph replay. 64 sequences, contexts 256 + U[0, 128] in a paged KV pool of
16-token blocks (permuted block tables, N(0, 1) bf16 contents); random N(0, 0.02) bf16 weights,
every decoder linear int8 per output channel, tied bf16 LM head.

Other workloads (each prints its own JSON line):
  linear     one int8 linear [3072 x 1024] (Qwen3-0.6B gate_proj) on 16 tokens -> GB/s
  attention  paged-attention decode, 64 sequences, contexts U[128, 2048], 16 q / 8 KV heads -> GB/s
  prefill    chunked-prefill step: one 1984-token prompt chunk + 64 decodes (contexts U[64, 1024])
             on the same 0.6B model -> tok/s
  decode8b   Qwen3-8B-shaped int8 decode, 256 tokens, contexts U[512, 4096] -> tok/s
  sample     temperature / top-k / top-p sampling of 64 rows of 151936 logits -> rows/s

Every line carries ``roofline`` for the workload's dominant kernel (algorithmic bytes or flops per
launch / its average duration, HIP events on the launch stream, inputs rotated past the 256 MB
Infinity Cache) and ``cpu_baseline``: the CPU oracle (a PyTorch restatement of the reference's
path) timed on this host's cores on a bounded sample of the same workload.
"""

from __future__ import annotations

import argparse
import json
import os
import platform
import random
import sys
import time
from pathlib import Path

ROOT = Path(__file__).resolve().parent
sys.path.insert(0, str(ROOT))

METRIC = "decode tok/s at batch 64 (Qwen3-0.6B int8); int8 GEMV + attn HBM GB/s vs peak"
HBM_PEAK_GBS = 8000.0
MFMA_BF16_PEAK_TFLOPS = 2500.0
BATCH, CTX_LO, CTX_HI = 64, 256, 384
# FETCH_SIZE x 2.0 + WRITE_SIZE x 1.0 of one fused decode-attention launch on the decode workload,
# from rocprofv3 --pmc: 42,870.85 KiB x 2 x 1024 + 512 KiB x 1024
# (profiles/paged_decode_kernel_traffic_pmc.md).
ATTN_TRAFFIC_BYTES: int | None = 88_323_789
# The same counters over one layer's four decode linears, summed, and over one launch of the
# single linear and of paged attention at 64 sequences x U[128, 2048]
# (profiles/decode_linears_and_attention_traffic_pmc.md).
LINEAR_TRAFFIC_BYTES: int | None = 25_903_104
CONFIG1_TRAFFIC_BYTES: int | None = 3_589_120
CONFIG2_TRAFFIC_BYTES: int | None = 279_336_320


def log(msg: str) -> None:
    print(f"[bench] {msg}", file=sys.stderr, flush=True)


def cpu_threads() -> int:
    """Every core this process may run on (its CPU affinity)."""
    return len(os.sched_getaffinity(0))


def cpu_model() -> str:
    """The host CPU's model name as ``lscpu`` prints it."""
    import subprocess

    try:
        out = subprocess.run(["lscpu"], capture_output=True, text=True, timeout=10, check=True).stdout
        for ln in out.splitlines():
            if ln.strip().startswith("Model name:"):
                return ln.split(":", 1)[1].strip()
    except (OSError, subprocess.SubprocessError):
        pass
    try:
        for ln in Path("/proc/cpuinfo").read_text().splitlines():
            if ln.startswith("model name"):
                return ln.split(":", 1)[1].strip()
    except OSError:
        pass
    return platform.processor() or platform.machine()


def hip_time(launch, count: int, reps: int = 5) -> float:
    """Seconds per launch: ``launch(i)`` for i < count queued back to back behind a spin kernel
    (long enough for the host to queue them all), bracketed by HIP events on the current stream
    (the stream the kernels are launched on); the median over passes of each pass's mean, after
    one warm-up pass, with at least ``reps`` passes and at least 100 timed launches in all."""
    import torch

    for i in range(count):
        launch(i)
    torch.cuda.synchronize()
    passes = max(reps, -(-100 // count))
    times = []
    for _ in range(passes):
        e0, e1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        torch.cuda._sleep(max(5_000_000, 250_000 * count))
        e0.record()
        for i in range(count):
            launch(i)
        e1.record()
        torch.cuda.synchronize()
        times.append(e0.elapsed_time(e1) * 1e-3 / count)
    times.sort()
    return times[len(times) // 2]


def decode_kernel_name(group: int, partition_tokens: int, fused: bool) -> str:
    """The decode-attention instantiation the C ABI launches (attention.hip:launch_decode): the
    fused decode-step entry point always four wavefronts; the plain one eight for splits of 1024+
    keys when the group has at most two query heads."""
    waves = 8 if (not fused and group <= 2 and partition_tokens >= 1024) else 4
    return f"paged_decode_kernel<{group}, {waves}, {'true' if fused else 'false'}, false>"


def dec_linear_name(m: int, k: int, epilogue: int, norm: bool) -> str:
    """The decode-linear instantiation msa_int8_linear_dec launches (gemv_dec.hip:dec_shape)."""
    kw = k // 256
    if epilogue == 1:
        nt, mt = (4 if kw <= 8 else 2), (2 if m > 16 and kw <= 8 else 1)
    elif epilogue == 0:
        nt, mt = (2 if m > 16 else 1), (2 if m > 16 and kw <= 8 else 1)
    else:
        nt, mt = 1, 1
    return f"dec_linear_kernel<{nt}, {mt}, {kw}, 4, {1 if norm else 0}, {epilogue}>"


def cpu_time(fn, budget_s: float = 20.0, max_reps: int = 5, min_reps: int = 5) -> tuple[float, int]:
    """Median seconds of ``fn()`` on the host after two warm-ups, at least ``min_reps`` runs and as
    many more (up to ``max_reps``) as fit the budget."""
    fn()
    t = time.perf_counter()
    fn()
    first = time.perf_counter() - t
    reps = max(min_reps, min(max_reps, int(budget_s / max(first, 1e-6))))
    times = []
    for _ in range(reps):
        t = time.perf_counter()
        fn()
        times.append(time.perf_counter() - t)
    times.sort()
    return times[len(times) // 2], reps


def cpu_fields(value: float, unit: str, sample: str) -> dict:
    import torch

    return {"value": round(value, 3), "unit": unit, "cores": torch.get_num_threads(), "kind": "port", "sample": sample,
            "cpu": cpu_model(), "torch": torch.__version__}


def roofline(kernel: str, bound: str, achieved: float, per_launch: int, secs: float, traffic=None) -> dict:
    peak, unit = (HBM_PEAK_GBS, "GB/s") if bound == "hbm" else (MFMA_BF16_PEAK_TFLOPS, "TFLOP/s")
    out = {"kernel": kernel, "bound": bound, "achieved": round(achieved, 1), "peak": peak, "unit": unit,
           "frac": round(achieved / peak, 4), "traffic": traffic, "us_per_launch": round(secs * 1e6, 3)}
    out["bytes_per_launch" if bound == "hbm" else "flops_per_launch"] = per_launch
    return out


def line(metric: str, value: float, unit: str, args, ms: float, config: dict, higher: bool = True) -> dict:
    return {"metric": metric, "value": round(value, 1), "unit": unit, "n_gpus": 1, "steps": args.steps,
            "warmup": args.warmup, "ms_per_step": round(ms, 4), "higher_is_better": higher, "scaling": "weak",
            "vs_baseline": None, "dtype": "bf16", "data": "synthetic", "config": config}


# ---- algorithmic work per unit ---------------------------------------------------------------------


def attention_bytes(ctx: list[int], heads: int, kv_heads: int, dim: int) -> int:
    """One decode-attention launch: every context token's K and V for every KV head, the queries
    and outputs, the block-table entries read and the per-sequence ints."""
    kv = 2 * kv_heads * dim * 2 * sum(ctx)
    qo = 2 * len(ctx) * heads * dim * 2
    tables = 4 * sum(-(-c // 16) for c in ctx)
    return kv + qo + tables + 8 * len(ctx)


def attention_qkv_bytes(ctx: list[int], heads: int, kv_heads: int, dim: int) -> int:
    """One fused decode-attention launch (per-head norms, RoPE, KV write, attention): the cached K and
    V of every earlier context token for every KV head, each sequence's qkv projection row, its new
    key and value written to the cache, its outputs, the rotary rows of its position (float32 cos
    and sin), the block-table entries read and the per-sequence ints."""
    kv = 2 * kv_heads * dim * 2 * sum(c - 1 for c in ctx)
    rows = len(ctx) * ((heads + 2 * kv_heads) * dim * 2 + 2 * kv_heads * dim * 2 + heads * dim * 2 + 2 * dim * 4)
    tables = 4 * sum(-(-c // 16) for c in ctx)
    return kv + rows + tables + 16 * len(ctx)


def linear_bytes(m: int, n: int, k: int) -> int:
    """One int8 linear: int8 weights, bf16 scales, bf16 x in, bf16 y out."""
    return n * k + 2 * n + 2 * m * k + 2 * m * n


# ---- shared model setup -----------------------------------------------------------------------------


def build_int8_model(cfg: dict, seed: int, dev, max_positions: int, on_device: bool = False):
    from miniserve_amd import workloads
    from miniserve_amd.quant.int8 import quantize_int8_

    weights = workloads.random_weights(cfg, seed=seed, device="cuda" if on_device else "cpu")
    model = workloads.build_model(cfg, weights, dev, max_positions=max_positions)
    quantize_int8_(model)
    return model, weights


def decode_sched(cfg: dict, batch, seed: int):
    from miniserve_amd.runner.model_runner import ScheduledChunk

    rng = random.Random(seed)
    sched = []
    for c, table, tok in zip(batch.context_lens, batch.block_tables, batch.token_ids, strict=True):
        sched.append(ScheduledChunk([rng.randrange(cfg["vocab_size"]) for _ in range(c - 1)] + [tok], c - 1, 1, table))
    return sched


def time_layer_attention(runner, sched, cfg, fused: bool = True) -> tuple[float, int, str]:
    """The dominant decode kernel as the step runs it -- ``fused``: per-head q/k-norm, RoPE, KV write
    and attention from the qkv projection rows (the token-split decode step); else attention from
    normed, rotated q after a separate cache write (larger batches) -- one launch per layer
    (distinct KV pools) per pass on the step's own metadata; returns (seconds per launch,
    algorithmic bytes per launch, kernel name)."""
    import torch

    from miniserve_amd import kernels
    from miniserve_amd.model.layers import RotaryEmbedding

    inp = runner.prepare(sched)
    d = inp.attn.decode
    dev = runner.device
    heads, kvh, dim = cfg["num_attention_heads"], cfg["num_key_value_heads"], cfg["head_dim"]
    ptok, parts = kernels.decode_plan(d.num_seqs, kvh, d.block_tables.shape[1], heads // kvh, d.split_context)
    g = torch.Generator(device=dev).manual_seed(5)
    out = torch.empty(len(sched), heads, dim, dtype=torch.bfloat16, device=dev)
    caches = runner.kv_caches
    ctx = [s.num_computed + 1 for s in sched]
    if not fused:
        q = torch.randn(len(sched), heads, dim, device=dev, generator=g).to(torch.bfloat16)

        def launch_plain(i):
            kc, vc = caches[i]
            kernels.paged_attention_decode(q, kc, vc, d.block_tables, d.context_lens, d.q_rows, ptok, parts,
                                           dim**-0.5, out)

        secs = hip_time(launch_plain, len(caches))
        return secs, attention_bytes(ctx, heads, kvh, dim), decode_kernel_name(heads // kvh, ptok, False)
    qkv = torch.randn(len(sched), (heads + 2 * kvh) * dim, device=dev, generator=g).to(torch.bfloat16)
    model = getattr(runner, "model", None)
    if model is not None:
        cos_t, sin_t = model.rotary.cos, model.rotary.sin
        norms = [(ly.self_attn.q_norm.weight, ly.self_attn.k_norm.weight) for ly in model.layers]
    else:  # the kernel-only entry point has no model: the same tables, unit norm weights
        rot = RotaryEmbedding(dim, max(ctx) + 1, cfg["rope_theta"])
        rot.build(dev)
        cos_t, sin_t = rot.cos, rot.sin
        ones = torch.ones(dim, dtype=torch.bfloat16, device=dev)
        norms = [(ones, ones)] * len(caches)

    def launch(i):
        kc, vc = caches[i]
        qw, kw = norms[i]
        kernels.paged_attention_decode_qkv(qkv, heads, qw, kw, cfg["rms_norm_eps"], cos_t, sin_t,
                                           inp.attn.slot_mapping, kc, vc, d.block_tables, d.context_lens, d.q_rows,
                                           ptok, parts, dim**-0.5, out)

    secs = hip_time(launch, len(caches))
    return secs, attention_qkv_bytes(ctx, heads, kvh, dim), decode_kernel_name(heads // kvh, ptok, True)


def decode_linear_bytes(m: int, n: int, k: int, epilogue: int, norm: bool) -> int:
    """One decode-step linear as it runs in the step: int8 weights, bf16 row scales, bf16 x in, bf16 y
    out (n / 2 columns after silu * up), plus the residual read of a residual epilogue and the
    RMSNorm weights of a norm prologue."""
    from miniserve_amd import kernels

    cols = n // 2 if epilogue == kernels.EPI_SILU_MUL else n
    extra = (2 * m * n if epilogue == kernels.EPI_RESIDUAL else 0) + (2 * k if norm else 0)
    return n * k + 2 * n + 2 * m * k + 2 * m * cols + extra


def time_layer_linears(model, tokens: int, dev) -> list[tuple[str, float, int, str]]:
    """The four int8 decode linears of a layer as the decode step runs them (the decode-linear kernel
    with the step's prologues and epilogues, ``tokens`` activation rows), each timed over one launch
    per layer on that layer's own weights (28 x 18 MB, more than the Infinity Cache holds); returns
    (name, seconds per launch, algorithmic bytes per launch, kernel) per linear."""
    import torch

    from miniserve_amd import kernels

    cfg = model.cfg
    h, qsz, inter = cfg.hidden_size, cfg.num_attention_heads * cfg.head_dim, cfg.intermediate_size
    g = torch.Generator(device=dev).manual_seed(11)
    x = torch.randn(tokens, h, generator=g, device=dev).to(torch.bfloat16)
    a = torch.randn(tokens, qsz, generator=g, device=dev).to(torch.bfloat16)
    act = torch.randn(tokens, inter, generator=g, device=dev).to(torch.bfloat16)
    res = torch.randn(tokens, h, generator=g, device=dev).to(torch.bfloat16)
    layers = model.layers
    out = []

    def qkv(i):
        ly = layers[i]
        kernels.int8_linear_dec(x, ly.self_attn.qkv_proj.qweight, ly.self_attn.qkv_proj.kscale,
                                norm_w=ly.input_layernorm.weight, eps=cfg.rms_norm_eps)

    def o(i):
        p = layers[i].self_attn.o_proj
        kernels.int8_linear_dec(a, p.qweight, p.kscale, kernels.EPI_RESIDUAL, residual=res, out=res)

    def gate_up(i):
        ly = layers[i]
        kernels.int8_linear_dec(x, ly.mlp.gate_up_proj.qweight, ly.mlp.gate_up_proj.kscale, kernels.EPI_SILU_MUL,
                                norm_w=ly.post_attention_layernorm.weight, eps=cfg.rms_norm_eps)

    def down(i):
        p = layers[i].mlp.down_proj
        kernels.int8_linear_dec(act, p.qweight, p.kscale, kernels.EPI_RESIDUAL, residual=res, out=res)

    for name, fn, n, k, epi, norm in (
        ("qkv + input RMSNorm", qkv, qsz + 2 * cfg.num_key_value_heads * cfg.head_dim, h, kernels.EPI_NONE, True),
        ("o + residual", o, h, qsz, kernels.EPI_RESIDUAL, False),
        ("gate_up + RMSNorm + silu*up", gate_up, 2 * inter, h, kernels.EPI_SILU_MUL, True),
        ("down + residual", down, h, inter, kernels.EPI_RESIDUAL, False),
    ):
        secs = hip_time(fn, len(layers))
        out.append((name, secs, decode_linear_bytes(tokens, n, k, epi, norm), dec_linear_name(tokens, k, epi, norm)))
    return out


def copy_bandwidth(dev) -> float:
    """GB/s of a 512 MiB device copy counted as 2x its bytes, the median of 5 runs of 20 copies
    after 3 warm-up copies (the reference's measurement, bench/bandwidth.py:21-34)."""
    import torch

    x = torch.empty(256 << 20, dtype=torch.bfloat16, device=dev)
    y = torch.empty_like(x)
    runs = []
    for _ in range(5):
        for _ in range(3):
            y.copy_(x)
        torch.cuda.synchronize()
        t = time.perf_counter()
        for _ in range(20):
            y.copy_(x)
        torch.cuda.synchronize()
        runs.append(2 * x.numel() * 2 * 20 / (time.perf_counter() - t) / 1e9)
    del x, y
    torch.cuda.empty_cache()
    return sorted(runs)[2]


def time_graph_steps(runner, sched, steps: int, warmup: int) -> float:
    import torch

    for _ in range(warmup):
        runner.execute(sched)
    torch.cuda.synchronize()
    t = time.perf_counter()
    for _ in range(steps):
        runner.execute(sched)
    torch.cuda.synchronize()
    return (time.perf_counter() - t) / steps


# ---- workloads ------------------------------------------------------------------------------------


def bench_decode(args) -> dict:
    import torch

    from miniserve_amd import workloads
    from miniserve_amd.runner.model_runner import ModelRunner

    dev = torch.device("cuda:0")
    cfg = workloads.QWEN3_0_6B
    t0 = time.time()
    model, weights = build_int8_model(cfg, args.seed, dev, 4096)
    batch = workloads.decode_batch(BATCH, CTX_LO, CTX_HI, seed=args.seed + 1, vocab=cfg["vocab_size"], spare_blocks=64)
    runner = ModelRunner(model, dev, use_graphs=True, max_model_len=4096)
    runner.allocate_kv_cache(batch.num_blocks)
    workloads.fill_kv_pool_(runner.kv_cache, seed=args.seed + 2, on_device=True)
    sched = decode_sched(cfg, batch, args.seed + 3)
    torch.cuda.synchronize()
    log(f"setup {time.time() - t0:.1f}s: 28-layer int8 model, {batch.num_blocks} KV blocks")

    def eager_step() -> list[int]:
        return runner.forward_greedy(runner.prepare(sched)).tolist()

    for _ in range(2):
        eager_step()
    torch.cuda.synchronize()
    t = time.perf_counter()
    n_eager = max(3, args.steps // 4)
    for _ in range(n_eager):
        eager_step()
    torch.cuda.synchronize()
    eager_dt = (time.perf_counter() - t) / n_eager
    graph_ids = runner.execute(sched)
    if [g[0] for g in graph_ids] != eager_step():
        raise RuntimeError("captured decode step disagrees with the eager step")
    dt = time_graph_steps(runner, sched, args.steps, args.warmup)
    # The device side of the same step: the captured graph replayed back to back (same inputs),
    # HIP events on its stream; the step above adds the host's preparation, upload and sync.
    cap = runner.graphs[len(sched)]
    with torch.cuda.stream(cap.stream):
        e0, e1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        e0.record()
        for _ in range(args.steps):
            cap.graph.replay()
        e1.record()
    torch.cuda.synchronize()
    replay_ms = e0.elapsed_time(e1) / args.steps
    log(f"eager {eager_dt * 1e3:.3f} ms/step; graph {args.steps} steps: {dt * 1e3:.3f} ms/step, {BATCH / dt:.0f} tok/s; "
        f"graph replay alone {replay_ms:.3f} ms")
    secs, nbytes, kname = time_layer_attention(runner, sched, cfg)
    log(f"decode attention: {secs * 1e6:.2f} us/launch, {nbytes / secs / 1e9:.0f} GB/s")
    out = line(METRIC, BATCH / dt, "tok/s", args, dt * 1e3, {
        "workload": "Qwen3-0.6B-architecture int8 decode step (28 layers, random init)",
        "batch": BATCH, "context": f"{CTX_LO}+U[0,{CTX_HI - CTX_LO}]", "sum_context": sum(batch.context_lens),
        "kv_block": 16, "weights": "int8 per-output-channel, bf16 activations, fp32 accumulation, tied bf16 LM head",
        "parallelism": "none", "hip_graph": True, "eager_ms_per_step": round(eager_dt * 1e3, 4),
        "graph_replay_ms": round(replay_ms, 4)})
    out["roofline"] = roofline(kname, "hbm", nbytes / secs / 1e9, nbytes, secs, ATTN_TRAFFIC_BYTES)
    # The other half of the metric: the four int8 decode linears of a layer, their algorithmic bytes
    # over their summed kernel time.
    lins = time_layer_linears(model, BATCH, dev)
    lin_secs, lin_bytes = sum(t for _, t, _, _ in lins), sum(b for _, _, b, _ in lins)
    for name, t, b, kn in lins:
        log(f"decode linear {name} ({kn}): {t * 1e6:.2f} us/launch, {b / t / 1e9:.0f} GB/s")
    out["roofline_gemv"] = roofline("dec_linear_kernel (qkv, o, gate_up, down of one layer)", "hbm",
                                    lin_bytes / lin_secs / 1e9, lin_bytes, lin_secs)
    out["roofline_gemv"]["per_linear_us"] = {name: round(t * 1e6, 3) for name, t, _, _ in lins}
    out["roofline_gemv"]["kernels"] = {name: kn for name, _, _, kn in lins}
    out["roofline_gemv"]["traffic"] = LINEAR_TRAFFIC_BYTES
    # The metric's GEMV and attention at their own workloads: the single int8 linear through
    # Int8Linear.forward, and paged-attention decode at 64 sequences x U[128, 2048].
    lins, x1 = setup_config1(dev, args.seed + 10)
    secs1, bytes1, kname1 = time_config1(lins, x1)
    log(f"int8 linear [3072x1024] x 16 (Int8Linear.forward): {secs1 * 1e6:.2f} us, {bytes1 / secs1 / 1e9:.0f} GB/s")
    out["roofline_config1"] = roofline(kname1, "hbm", bytes1 / secs1 / 1e9, bytes1, secs1, CONFIG1_TRAFFIC_BYTES)
    out["roofline_config1"]["workload"] = "Int8Linear.forward, W [3072x1024] int8, x [16x1024] bf16"
    del lins, x1
    q2, _, _, kv2, _, _, meta2, ctx2 = setup_config2(dev, args.seed + 20)
    secs2, bytes2, kname2 = time_config2(q2, kv2, meta2, ctx2)
    log(f"paged decode attention, 64 seqs x U[128,2048]: {secs2 * 1e6:.2f} us, {bytes2 / secs2 / 1e9:.0f} GB/s")
    out["roofline_config2"] = roofline(kname2, "hbm", bytes2 / secs2 / 1e9, bytes2, secs2, CONFIG2_TRAFFIC_BYTES)
    out["roofline_config2"]["workload"] = "paged-attention decode, 64 seqs, ctx U[128,2048], 16q/8kv, d=128"
    del q2, kv2, meta2
    torch.cuda.empty_cache()
    copy = copy_bandwidth(dev)
    log(f"copy bandwidth (512 MiB, 2x bytes): {copy:.0f} GB/s")
    out["copy_bandwidth"] = {"value": round(copy, 1), "unit": "GB/s", "frac_of_peak": round(copy / HBM_PEAK_GBS, 4),
                             "method": "512 MiB device copy x 20, 2x bytes, median of 5"}
    for key in ("roofline", "roofline_gemv", "roofline_config1", "roofline_config2"):
        out[key]["frac_of_copy_bw"] = round(out[key]["achieved"] / copy, 4)
    if not args.no_cpu_baseline:
        from oracle import model as om

        torch.set_num_threads(cpu_threads())
        ocfg = om.Config.from_dict(cfg)
        ow = om.quantize_weights(weights, ocfg)
        okv = [(kc.cpu(), vc.cpu()) for kc, vc in runner.kv_caches]
        tables = om.tables_for(ocfg, 4096)
        step = om.prepare([(s.token_ids, s.num_computed, s.num_new, s.block_table) for s in sched], 16)
        med, reps = cpu_time(lambda: om.run_step(ocfg, ow, okv, step, 16, tables))
        log(f"cpu oracle: {med:.3f} s/step on {cpu_threads()} threads")
        out["cpu_baseline"] = cpu_fields(BATCH / med, "tok/s", "the full decode step (64 tokens, 28 layers, LM head, "
                                         f"argmax), median of {reps} after 2 warm-ups")
    return out


def setup_config1(dev, seed: int):
    """The single int8 linear workload through the reference's module API: ``Int8Linear(W)`` for
    W ~ N(0, 0.02) bf16 [3072 x 1024] (Qwen3-0.6B gate_proj), enough distinct copies to exceed
    the 256 MB Infinity Cache, and x ~ N(0, 1) bf16 [16 x 1024]."""
    import torch

    from miniserve_amd.quant.int8 import Int8Linear

    m, n, k = 16, 3072, 1024
    copies = -(-(300 << 20) // (n * k))
    g = torch.Generator(device=dev).manual_seed(seed)
    lins = [Int8Linear((torch.randn(n, k, generator=g, device=dev) * 0.02).to(torch.bfloat16)) for _ in range(copies)]
    x = torch.randn(m, k, generator=g, device=dev).to(torch.bfloat16)
    return lins, x


def time_config1(lins, x) -> tuple[float, int, str]:
    """(seconds per ``Int8Linear.forward`` call, algorithmic bytes per call, kernel), one call per
    weight copy per pass."""
    m, k = x.shape
    n = lins[0].out_features
    secs = hip_time(lambda i: lins[i](x), len(lins))
    return secs, linear_bytes(m, n, k), dec_linear_name(m, k, 0, False)


def bench_linear(args) -> dict:
    import torch

    dev = torch.device("cuda:0")
    lins, x = setup_config1(dev, args.seed)
    secs, nbytes, kname = time_config1(lins, x)
    m, k = x.shape
    n = lins[0].out_features
    gbs = nbytes / secs / 1e9
    log(f"int8 linear [{n}x{k}] x {m}: {secs * 1e6:.2f} us/launch, {gbs:.0f} GB/s")
    out = line("int8 linear [3072x1024] x 16 tokens: algorithmic HBM GB/s", gbs, "GB/s", args, secs * 1e3, {
        "workload": "single int8 weight-only linear, Qwen3-0.6B gate_proj shape, through Int8Linear.forward",
        "tokens": m, "out_features": n, "in_features": k, "weights": "N(0,0.02) bf16 quantized per output channel",
        "copies_rotated": len(lins)})
    out["roofline"] = roofline(kname, "hbm", gbs, nbytes, secs)
    if not args.no_cpu_baseline:
        from oracle import int8 as oi

        torch.set_num_threads(cpu_threads())
        xc, qc, sc = x.cpu(), lins[0].qweight.cpu(), lins[0].scale.cpu()
        med, reps = cpu_time(lambda: oi.int8_linear(xc, qc, sc), budget_s=10.0, max_reps=200)
        out["cpu_baseline"] = cpu_fields(nbytes / med / 1e9, "GB/s", f"the same linear on the CPU oracle (whole-matrix "
                                         f"dequantization + F.linear), median of {reps}")
    return out


ATTN_POOLS = 4  # 4 x ~286 MB of K/V: repeats cannot come from the Infinity Cache


def setup_config2(dev, seed: int):
    """The paged-attention decode workload: 64 sequences, contexts U[128, 2048], 16 q / 8 KV heads,
    head_dim 128, N(0, 1) bf16 q / new k, v / pools, block tables slices of one permutation of the
    pool's blocks; ATTN_POOLS pools, rotated per call. Returns (q, knew, vnew, kv, slots, chunks,
    meta, context lengths)."""
    import torch

    from miniserve_amd import workloads
    from miniserve_amd.attention import backends as hb

    nseq, heads, kvh, dim = 64, 16, 8, 128
    b = workloads.decode_batch(nseq, 128, 2048, seed=seed + 1, spare_blocks=0)
    kv = torch.empty(ATTN_POOLS, 2, b.num_blocks * 16, kvh, dim, dtype=torch.bfloat16, device=dev)
    workloads.fill_kv_pool_(kv, seed=seed + 2, on_device=True)
    g = torch.Generator(device=dev).manual_seed(seed + 3)
    q = torch.randn(nseq, heads, dim, generator=g, device=dev).to(torch.bfloat16)
    knew = torch.randn(nseq, kvh, dim, generator=g, device=dev).to(torch.bfloat16)
    vnew = torch.randn(nseq, kvh, dim, generator=g, device=dev).to(torch.bfloat16)
    slots = torch.tensor(b.slot_mapping, dtype=torch.int64, device=dev)
    chunks = [hb.SeqChunk(i, 1, c - 1, t) for i, (c, t) in enumerate(zip(b.context_lens, b.block_tables, strict=True))]
    meta = hb.build_attention_metadata(chunks, slots, 16)
    return q, knew, vnew, kv, slots, chunks, meta, b.context_lens


def time_config2(q, kv, meta, ctx) -> tuple[float, int, str]:
    """(seconds per decode-attention launch, algorithmic bytes per launch, kernel) on the plain
    decode entry point, one launch per pool per pass."""
    import torch

    from miniserve_amd import kernels

    heads, kvh, dim = q.shape[1], kv.shape[3], q.shape[2]
    d = meta.decode
    ptok, parts = kernels.decode_plan(d.num_seqs, kvh, d.block_tables.shape[1], heads // kvh, d.split_context)
    out_t = torch.empty_like(q)

    def kern(i):
        kernels.paged_attention_decode(q, kv[i % ATTN_POOLS, 0], kv[i % ATTN_POOLS, 1], d.block_tables, d.context_lens,
                                       d.q_rows, ptok, parts, dim**-0.5, out_t)

    secs = hip_time(kern, 2 * ATTN_POOLS)
    return secs, attention_bytes(ctx, heads, kvh, dim), decode_kernel_name(heads // kvh, ptok, False)


def bench_attention(args) -> dict:
    import torch

    from miniserve_amd.attention import backends as hb

    dev = torch.device("cuda:0")
    q, knew, vnew, kv, slots, chunks, meta, ctx = setup_config2(dev, args.seed)
    nseq, heads, dim = q.shape
    kvh = kv.shape[3]
    scale = dim**-0.5

    def op(i):
        hb.paged_attention(q, knew, vnew, kv[i % ATTN_POOLS, 0], kv[i % ATTN_POOLS, 1], meta, scale)

    op_secs = hip_time(op, 2 * ATTN_POOLS)
    op_bytes = 4096 * sum(ctx) + 786_432 + 4 * sum(-(-c // 16) for c in ctx) + 256
    k_secs, k_bytes, kname = time_config2(q, kv, meta, ctx)
    log(f"paged_attention (write + attend): {op_secs * 1e6:.2f} us, {op_bytes / op_secs / 1e9:.0f} GB/s; "
        f"decode kernel {k_secs * 1e6:.2f} us, {k_bytes / k_secs / 1e9:.0f} GB/s")
    out = line("paged-attention decode GB/s (64 seqs, ctx U[128,2048], 16q/8kv, d=128)", op_bytes / op_secs / 1e9,
               "GB/s", args, op_secs * 1e3, {
                   "workload": "paged_attention: KV write + decode attention through permuted 16-token block tables",
                   "seqs": nseq, "sum_context": sum(ctx), "heads": heads, "kv_heads": kvh, "head_dim": dim,
                   "bytes_per_call": op_bytes, "pools_rotated": ATTN_POOLS})
    out["roofline"] = roofline(kname, "hbm", k_bytes / k_secs / 1e9, k_bytes, k_secs)
    if not args.no_cpu_baseline:
        from oracle import attention as oa

        torch.set_num_threads(cpu_threads())
        kc, vc = kv[0, 0].cpu(), kv[0, 1].cpu()
        qc, kn, vn, sl = q.cpu(), knew.cpu(), vnew.cpu(), slots.cpu()
        ometa = oa.build_attention_metadata([oa.SeqChunk(*c.__dict__.values()) for c in chunks], sl, 16)
        med, reps = cpu_time(lambda: oa.paged_attention(qc, kn, vn, kc, vc, ometa, scale), budget_s=20.0)
        out["cpu_baseline"] = cpu_fields(op_bytes / med / 1e9, "GB/s", f"the same paged_attention call on the CPU "
                                         f"oracle (gather + SDPA), median of {reps}")
    return out


LONG_CONTEXT_CASES = ((1, 32768, 32768), (4, 32768, 32768), (16, 16384, 32768))


def bench_long_context(args) -> dict:
    """Decode attention at small batches and long contexts, the plain decode entry point: 1 and 4
    sequences at 32,768 keys and 16 at U[16384, 32768], 16 q / 8 KV heads, head_dim 128, N(0, 1)
    bf16, block tables slices of one permutation of the pool. Splits are keyed to the 32K planned
    context (at most 32 per sequence), so these launches run split partials and the split merge.
    The line reports 16 sequences; the other batch sizes sit under ``sweep``."""
    import torch

    from miniserve_amd import kernels, workloads
    from miniserve_amd.attention import backends as hb

    dev = torch.device("cuda:0")
    heads, kvh, dim, pools = 16, 8, 128, 2  # 2 pools x 2.1 GB at batch 16: past the 256 MB Infinity Cache
    sweep = {}
    for nseq, lo, hi in LONG_CONTEXT_CASES:
        b = workloads.decode_batch(nseq, lo, hi, seed=args.seed + nseq, spare_blocks=0)
        kv = torch.empty(pools, 2, b.num_blocks * 16, kvh, dim, dtype=torch.bfloat16, device=dev)
        workloads.fill_kv_pool_(kv, seed=args.seed + 2, on_device=True)
        g = torch.Generator(device=dev).manual_seed(args.seed + 3)
        q = torch.randn(nseq, heads, dim, generator=g, device=dev).to(torch.bfloat16)
        slots = torch.tensor(b.slot_mapping, dtype=torch.int64, device=dev)
        chunks = [hb.SeqChunk(i, 1, c - 1, t) for i, (c, t) in enumerate(zip(b.context_lens, b.block_tables,
                                                                            strict=True))]
        meta = hb.build_attention_metadata(chunks, slots, 16)
        d = meta.decode
        ptok, parts = kernels.decode_plan(nseq, kvh, d.block_tables.shape[1], heads // kvh, 32768)
        out_t = torch.empty_like(q)

        def kern(i, kv=kv, q=q, d=d, ptok=ptok, parts=parts, out_t=out_t):
            kernels.paged_attention_decode(q, kv[i % pools, 0], kv[i % pools, 1], d.block_tables, d.context_lens,
                                           d.q_rows, ptok, parts, dim**-0.5, out_t)

        secs = hip_time(kern, 2 * pools)
        nbytes = attention_bytes(b.context_lens, heads, kvh, dim)
        used = max(-(-c // ptok) for c in b.context_lens)
        sweep[f"{nseq}x{lo}" if lo == hi else f"{nseq}xU[{lo},{hi}]"] = {
            "us_per_launch": round(secs * 1e6, 3), "gbs": round(nbytes / secs / 1e9, 1),
            "frac": round(nbytes / secs / 1e9 / HBM_PEAK_GBS, 4), "bytes_per_launch": nbytes,
            "split_tokens": ptok, "splits_per_longest_seq": used, "workgroups": nseq * kvh * parts,
            "partials_bytes": nseq * heads * parts * (dim + 2) * 4 if parts > 1 else 0,
            "kernel": decode_kernel_name(heads // kvh, ptok, False) + " + split merge"}
        log(f"decode attention {nseq} seqs x [{lo},{hi}] keys: {secs * 1e6:.2f} us, {nbytes / secs / 1e9:.0f} GB/s "
            f"({ptok}-key splits, {used} per longest sequence)")
        last = (nseq, lo, hi, secs, nbytes, ptok)
        del kv
        torch.cuda.empty_cache()
    nseq, lo, hi, secs, nbytes, ptok = last
    out = line(f"decode attention GB/s at small batch, long context ({nseq} seqs, ctx U[{lo},{hi}], 16q/8kv, d=128)",
               nbytes / secs / 1e9, "GB/s", args, secs * 1e3, {
                   "workload": "paged decode attention with split partials and merge, splits keyed to a 32K plan",
                   "seqs": nseq, "heads": heads, "kv_heads": kvh, "head_dim": dim, "pools_rotated": pools})
    out["roofline"] = roofline(decode_kernel_name(heads // kvh, ptok, False) + " + split merge", "hbm",
                               nbytes / secs / 1e9, nbytes, secs)
    out["sweep"] = sweep
    return out


def bench_prefill(args) -> dict:
    import torch

    from miniserve_amd import kernels, workloads
    from miniserve_amd.runner.model_runner import ModelRunner, ScheduledChunk

    dev = torch.device("cuda:0")
    cfg = workloads.QWEN3_0_6B
    model, weights = build_int8_model(cfg, args.seed, dev, 4096)
    dec = workloads.decode_batch(64, 64, 1024, seed=args.seed + 1, vocab=cfg["vocab_size"], spare_blocks=0)
    chunk = 1984
    pblocks = -(-chunk // 16)
    total_blocks = dec.num_blocks + pblocks
    runner = ModelRunner(model, dev, use_graphs=False, max_model_len=4096)
    runner.allocate_kv_cache(total_blocks)
    workloads.fill_kv_pool_(runner.kv_cache, seed=args.seed + 2, on_device=True)
    sched = decode_sched(cfg, dec, args.seed + 3)
    rng = random.Random(args.seed + 4)
    prompt = [rng.randrange(cfg["vocab_size"]) for _ in range(chunk)]
    sched.append(ScheduledChunk(prompt, 0, chunk, list(range(dec.num_blocks, total_blocks))))
    tokens = sum(s.num_new for s in sched)
    for _ in range(args.warmup):
        runner.execute(sched)
    torch.cuda.synchronize()
    t = time.perf_counter()
    for _ in range(args.steps):
        runner.execute(sched)
    torch.cuda.synchronize()
    dt = (time.perf_counter() - t) / args.steps
    log(f"chunked-prefill step ({tokens} tokens): {dt * 1e3:.3f} ms/step, {tokens / dt:.0f} tok/s")
    # dominant kernel: the gate_up GEMM at M = 2048 over the 28 layers' weights
    h = torch.randn(tokens, cfg["hidden_size"], device=dev).to(torch.bfloat16)
    y = torch.empty(tokens, cfg["intermediate_size"], dtype=torch.bfloat16, device=dev)
    lin = [layer.mlp.gate_up_proj for layer in model.layers]

    def launch(i):
        kernels.int8_linear(h, lin[i].qweight, lin[i].scale, kernels.EPI_SILU_MUL, out=y)

    secs = hip_time(launch, len(lin))
    flops = 2 * tokens * 2 * cfg["intermediate_size"] * cfg["hidden_size"]
    log(f"gate_up GEMM M={tokens}: {secs * 1e6:.1f} us, {flops / secs / 1e12:.1f} TFLOP/s")
    sum_dec = sum(dec.context_lens)
    step_flops = (2 * tokens * 15_728_640 * 28 + 4 * 16 * 128 * (chunk * (chunk + 1) // 2) * 28
                  + 8192 * sum_dec * 28 + 2 * 65 * 1024 * cfg["vocab_size"])
    out = line("chunked-prefill step tok/s (1984-token chunk + 64 decodes, Qwen3-0.6B int8)", tokens / dt, "tok/s", args,
               dt * 1e3, {"workload": "mixed flat batch: 64 decodes (contexts U[64,1024]) first, then one fresh "
                          "1984-token prompt chunk; eager step (prepare + forward + fused LM head/argmax + sync)",
                          "tokens": tokens, "step_tflop": round(step_flops / 1e12, 3),
                          "step_tflop_s": round(step_flops / dt / 1e12, 1)})
    # the step's largest kernel by time: the chunk's causal attention (the decode rows' attention
    # runs beside it on a second stream), timed alone over the 28 layers' KV pools
    from miniserve_amd.attention import backends as hb

    pslots = torch.tensor([dec.num_blocks * 16 + p for p in range(chunk)], device=dev)
    pmeta = hb.build_attention_metadata([hb.SeqChunk(0, chunk, 0, list(range(dec.num_blocks, total_blocks)))],
                                        pslots, 16)
    pq = torch.randn(chunk, 16, 128, device=dev).to(torch.bfloat16)
    caches = runner.kv_caches
    asecs = hip_time(lambda i: hb.attend(pq, caches[i][0], caches[i][1], pmeta, 128**-0.5), len(caches))
    aflops = 4 * 16 * 128 * (chunk * (chunk + 1) // 2)
    log(f"prefill attention (1984-token causal chunk): {asecs * 1e6:.1f} us, {aflops / asecs / 1e12:.1f} TFLOP/s")
    out["roofline"] = roofline("paged_prefill_kernel<2, true> (1984-token causal chunk, 16 q / 8 KV heads)", "mfma",
                               aflops / asecs / 1e12, aflops, asecs)
    out["roofline_gemm"] = roofline("int8_gemm256_kernel<192, 8, 2, 1> (gate_up + silu*up, M=2048, 256x192 tiles)", "mfma",
                                    flops / secs / 1e12, flops, secs)
    if not args.no_cpu_baseline:
        from oracle import model as om
        from oracle.attention import build_attention_metadata as oracle_meta

        torch.set_num_threads(cpu_threads())
        ocfg = om.Config.from_dict(cfg)
        ow = om.quantize_weights({k: v for k, v in weights.items() if k.startswith("layers.0.") or "layers." not in k},
                                 om.Config.from_dict({**cfg, "num_hidden_layers": 1}))
        step = om.prepare([(s.token_ids, s.num_computed, s.num_new, s.block_table) for s in sched], 16)
        ometa = oracle_meta(step.chunks, step.slot_mapping, 16)
        kc, vc = runner.kv_caches[0][0].cpu(), runner.kv_caches[0][1].cpu()
        tables = om.tables_for(ocfg, 4096)
        x0 = torch.nn.functional.embedding(step.input_ids, ow["embed_tokens.weight"])
        cos, sin = tables[0][step.positions], tables[1][step.positions]

        def one_layer():
            with torch.inference_mode():
                om.decoder_layer(ocfg, ow, 0, x0, cos, sin, kc, vc, ometa)

        def head():
            with torch.inference_mode():
                om.greedy(om.compute_logits(ocfg, ow, x0[step.logits_rows]))

        lay, reps = cpu_time(one_layer, budget_s=20.0, max_reps=3)
        hd, _ = cpu_time(head, budget_s=5.0, max_reps=3)
        est = 28 * lay + hd
        out["cpu_baseline"] = cpu_fields(tokens / est, "tok/s", f"one decoder layer of this step on the CPU oracle "
                                         f"(median of {reps}) x 28 + the LM head and argmax of its 65 sampled rows")
    return out


def bench_decode8b(args) -> dict:
    import torch

    from miniserve_amd import workloads
    from miniserve_amd.runner.model_runner import ModelRunner

    dev = torch.device("cuda:0")
    cfg = workloads.QWEN3_8B
    nseq = 256
    t0 = time.time()
    model, weights = build_int8_model(cfg, args.seed, dev, 4096 + 16, on_device=True)
    keep = {k: v.cpu() for k, v in weights.items() if k.startswith("layers.0.") or "layers." not in k}
    del weights
    torch.cuda.empty_cache()
    batch = workloads.decode_batch(nseq, 512, 4096, seed=args.seed + 1, vocab=cfg["vocab_size"], spare_blocks=0)
    runner = ModelRunner(model, dev, use_graphs=True, max_model_len=4096 + 16)
    runner.allocate_kv_cache(batch.num_blocks)
    workloads.fill_kv_pool_(runner.kv_cache, seed=args.seed + 2, on_device=True)
    sched = decode_sched(cfg, batch, args.seed + 3)
    torch.cuda.synchronize()
    log(f"setup {time.time() - t0:.1f}s: 36-layer 8B-shaped int8 model, {batch.num_blocks} KV blocks "
        f"({runner.kv_cache.numel() * 2 / 1e9:.1f} GB)")
    dt = time_graph_steps(runner, sched, args.steps, args.warmup)
    log(f"graph {args.steps} steps: {dt * 1e3:.3f} ms/step, {nseq / dt:.0f} tok/s")
    secs, nbytes, kname = time_layer_attention(runner, sched, cfg, fused=False)
    log(f"decode attention: {secs * 1e6:.2f} us/launch, {nbytes / secs / 1e9:.0f} GB/s")
    out = line("decode tok/s at batch 256 (Qwen3-8B-shaped int8, contexts U[512,4096])", nseq / dt, "tok/s", args,
               dt * 1e3, {"workload": "Qwen3-8B-architecture int8 decode step (36 layers, untied bf16 LM head, "
                          "random init)", "batch": nseq, "sum_context": sum(batch.context_lens), "kv_block": 16,
                          "hip_graph": True})
    out["roofline"] = roofline(kname, "hbm", nbytes / secs / 1e9, nbytes, secs)
    if not args.no_cpu_baseline:
        from oracle import model as om
        from oracle.attention import build_attention_metadata as oracle_meta

        torch.set_num_threads(cpu_threads())
        ocfg = om.Config.from_dict(cfg)
        ow = om.quantize_weights(keep, om.Config.from_dict({**cfg, "num_hidden_layers": 1}))
        step = om.prepare([(s.token_ids, s.num_computed, s.num_new, s.block_table) for s in sched], 16)
        ometa = oracle_meta(step.chunks, step.slot_mapping, 16)
        kc, vc = runner.kv_caches[0][0].cpu(), runner.kv_caches[0][1].cpu()
        tables = om.tables_for(ocfg, 4096 + 16)
        x0 = torch.nn.functional.embedding(step.input_ids, ow["embed_tokens.weight"])
        cos, sin = tables[0][step.positions], tables[1][step.positions]
        rows = 16  # LM-head sample: 16 of the 256 sampled rows, scaled by 16

        def one_layer():
            with torch.inference_mode():
                om.decoder_layer(ocfg, ow, 0, x0, cos, sin, kc, vc, ometa)

        def head():
            with torch.inference_mode():
                om.greedy(om.compute_logits(ocfg, ow, x0[:rows]))

        lay, reps = cpu_time(one_layer, budget_s=20.0, max_reps=3)
        hd, _ = cpu_time(head, budget_s=10.0, max_reps=3)
        est = 36 * lay + hd * (nseq / rows)
        out["cpu_baseline"] = cpu_fields(nseq / est, "tok/s", f"one decoder layer of this step on the CPU oracle "
                                         f"(median of {reps}) x 36 + the LM head/argmax of 16 rows x 16")
    return out


# ---- profiling entry points -----------------------------------------------------------------------


def kernel_only(mode: str, seed: int) -> int:
    """``single-linear`` / ``paged-attention``: the default line's single-linear and paged-attention
    fractions alone; ``attention``: only the decode-attention timing of the decode workload; ``linear``: the int8
    linears of the decode step (plus the single gate_proj-shaped linear) over rotated weights;
    ``step-linears``: the four decode linears of every layer of the 0.6B model as the decode step
    runs them; ``gemm``: the chunked-prefill step's gate_up GEMM at 2048 tokens over every layer's
    weights; ``prefill-attention``: its paged attention (a 1984-token chunk after 64 decodes) over
    28 KV pools; ``copy``: a 256 MiB copy, 10 times (a kernel of known traffic, to calibrate
    rocprofv3's FETCH_SIZE / WRITE_SIZE)."""
    import torch

    from miniserve_amd import kernels, workloads
    from miniserve_amd.runner.model_runner import ModelRunner

    dev = torch.device("cuda:0")
    if mode == "single-linear":  # Int8Linear.forward on [3072 x 1024] x 16 tokens over rotated weights
        lins, x = setup_config1(dev, seed)
        secs, nbytes, kname = time_config1(lins, x)
        print(json.dumps({"kernel": kname, "us_per_launch": round(secs * 1e6, 3), "bytes_per_launch": nbytes,
                          "GB_s": round(nbytes / secs / 1e9, 1), "copies": len(lins)}))
        return 0
    if mode == "paged-attention":  # decode attention, 64 sequences x U[128, 2048], rotated pools
        q, _, _, kv, _, _, meta, ctx = setup_config2(dev, seed)
        secs, nbytes, kname = time_config2(q, kv, meta, ctx)
        print(json.dumps({"kernel": kname, "us_per_launch": round(secs * 1e6, 3), "bytes_per_launch": nbytes,
                          "GB_s": round(nbytes / secs / 1e9, 1)}))
        return 0
    if mode == "copy":
        src = torch.empty(128 << 20, dtype=torch.bfloat16, device=dev).normal_()
        dst = torch.empty_like(src)
        for _ in range(10):
            dst.copy_(src)
        torch.cuda.synchronize()
        print(json.dumps({"copy_bytes_each_way": src.numel() * 2, "copies": 10}))
        return 0
    if mode == "step-linears":  # the four decode linears of every layer, as the decode step runs them
        model, _ = build_int8_model(workloads.QWEN3_0_6B, seed, dev, 4096, on_device=True)
        for name, t, b, kn in time_layer_linears(model, BATCH, dev):
            print(json.dumps({"linear": name, "kernel": kn, "us_per_launch": round(t * 1e6, 3),
                              "bytes_per_launch": b, "GB_s": round(b / t / 1e9, 1)}), flush=True)
        return 0
    if mode in ("gemm", "prefill-attention"):  # the chunked-prefill step's dominant kernels
        cfg = workloads.QWEN3_0_6B
        if mode == "gemm":
            model, _ = build_int8_model(cfg, seed, dev, 4096, on_device=True)
            h = torch.randn(2048, cfg["hidden_size"], device=dev).to(torch.bfloat16)
            y = torch.empty(2048, cfg["intermediate_size"], dtype=torch.bfloat16, device=dev)
            lin = [layer.mlp.gate_up_proj for layer in model.layers]
            secs = hip_time(lambda i: kernels.int8_linear(h, lin[i].qweight, lin[i].kscale, kernels.EPI_SILU_MUL,
                                                          out=y), len(lin))
            flops = 2 * 2048 * 2 * cfg["intermediate_size"] * cfg["hidden_size"]
            print(json.dumps({"kernel": "gate_up GEMM, M=2048", "us_per_launch": secs * 1e6,
                              "TFLOP_s": flops / secs / 1e12}))
            return 0
        from miniserve_amd.attention import backends as hb

        dec = workloads.decode_batch(64, 64, 1024, seed=seed + 1, spare_blocks=0)
        chunk = 1984
        blocks = dec.num_blocks + -(-chunk // 16)
        layers = 28
        kv = torch.empty(layers, 2, blocks * 16, 8, 128, dtype=torch.bfloat16, device=dev)
        workloads.fill_kv_pool_(kv, seed=seed + 2, on_device=True)
        chunks = [hb.SeqChunk(i, 1, c - 1, t) for i, (c, t) in enumerate(zip(dec.context_lens, dec.block_tables))]
        chunks.append(hb.SeqChunk(64, chunk, 0, list(range(dec.num_blocks, blocks))))
        slots = torch.tensor(dec.slot_mapping + [dec.num_blocks * 16 + p for p in range(chunk)], device=dev)
        meta = hb.build_attention_metadata(chunks, slots, 16)
        q = torch.randn(64 + chunk, 16, 128, device=dev).to(torch.bfloat16)
        secs = hip_time(lambda i: hb.attend(q, kv[i, 0], kv[i, 1], meta, 128**-0.5), layers)
        flops = 4 * 16 * 128 * (chunk * (chunk + 1) // 2) + 4 * 16 * 128 * sum(dec.context_lens)
        print(json.dumps({"kernel": "paged attention, 1984-token chunk + 64 decodes", "us_per_launch": secs * 1e6,
                          "TFLOP_s": flops / secs / 1e12}))
        return 0
    if mode == "linear":
        g = torch.Generator(device=dev).manual_seed(seed)
        shapes = [("gate_proj [3072x1024], 16 tokens", 16, 3072, 1024, kernels.EPI_NONE),
                  ("qkv [4096x1024] + q/k-norm/RoPE/cache, 64 tokens", 64, 4096, 1024, -1),
                  ("o [1024x2048] + residual, 64 tokens", 64, 1024, 2048, kernels.EPI_RESIDUAL),
                  ("gate_up [6144x1024] + norm + silu*up, 64 tokens", 64, 6144, 1024, kernels.EPI_SILU_MUL),
                  ("down [1024x3072] + residual, 64 tokens", 64, 1024, 3072, kernels.EPI_RESIDUAL),
                  # Qwen3-8B-shaped decode linears: weights large enough for a launch to stream at HBM rates
                  ("8B qkv [6144x4096], 16 tokens", 16, 6144, 4096, kernels.EPI_NONE),
                  ("8B o [4096x4096] + residual, 16 tokens", 16, 4096, 4096, kernels.EPI_RESIDUAL),
                  ("8B gate_up [24576x4096] + norm + silu*up, 16 tokens", 16, 24576, 4096, kernels.EPI_SILU_MUL),
                  ("8B gate_up [24576x4096] + norm + silu*up, 64 tokens", 64, 24576, 4096, kernels.EPI_SILU_MUL)]
        for name, m, n, k, epi in shapes:
            copies = max(8, -(-(300 << 20) // (n * k)))
            ws = torch.randint(-127, 128, (copies, n, k), dtype=torch.int8, device=dev, generator=g)
            sc = (torch.rand(copies, n, device=dev, generator=g) * 0.001).to(torch.bfloat16)
            x = torch.randn(m, k, device=dev, generator=g).to(torch.bfloat16)
            nw = torch.ones(k, dtype=torch.bfloat16, device=dev)
            resid = torch.randn(m, n, device=dev, generator=g).to(torch.bfloat16)
            y = torch.empty(m, n // 2 if epi == kernels.EPI_SILU_MUL else n, dtype=torch.bfloat16, device=dev)
            if epi == -1:
                pos = torch.arange(m, device=dev) + 300
                cos, sin = torch.randn(4096, 128, device=dev), torch.randn(4096, 128, device=dev)
                slots = torch.arange(m, device=dev)
                kc = torch.zeros(m, 8, 128, dtype=torch.bfloat16, device=dev)
                vc = torch.zeros_like(kc)

                def run(i):
                    kernels.qkv_rope_cache_rows(x, ws[i], sc[i], 16, 8, 128, nw[:128], nw[:128], 1e-6, pos, cos, sin,
                                                slots, kc, vc, norm_w=nw, eps=1e-6)
            elif epi == kernels.EPI_SILU_MUL:
                def run(i):
                    kernels.int8_linear_rows(x, ws[i], sc[i], epi, norm_w=nw, eps=1e-6, out=y)
            elif epi == kernels.EPI_RESIDUAL:
                def run(i):
                    kernels.int8_linear_rows(x, ws[i], sc[i], epi, residual=resid, out=y)
            else:
                def run(i):
                    kernels.int8_linear_rows(x, ws[i], sc[i], out=y)
            if epi == -1:
                def run_dec(i):
                    kernels.int8_linear_dec(x, ws[i], sc[i], norm_w=nw, eps=1e-6, out=y)
            elif epi == kernels.EPI_SILU_MUL:
                def run_dec(i):
                    kernels.int8_linear_dec(x, ws[i], sc[i], epi, norm_w=nw, eps=1e-6, out=y)
            elif epi == kernels.EPI_RESIDUAL:
                def run_dec(i):
                    kernels.int8_linear_dec(x, ws[i], sc[i], epi, residual=resid, out=y)
            else:
                def run_dec(i):
                    kernels.int8_linear_dec(x, ws[i], sc[i], out=y)
            runs = [("token-split rows kernel", run), ("decode kernel", run_dec)]
            nbytes = linear_bytes(m, n, k)
            for kind, fn in runs:
                secs = hip_time(fn, copies)
                label = name if not (epi == -1 and kind != "token-split rows kernel") else "qkv [4096x1024] + input norm, 64 tokens"
                print(json.dumps({"linear": label, "kernel": kind, "us_per_launch": round(secs * 1e6, 3),
                                  "bytes_per_launch": nbytes, "GB_s": round(nbytes / secs / 1e9, 1),
                                  "copies": copies}), flush=True)
            del ws, sc
        return 0
    cfg = workloads.QWEN3_0_6B
    batch = workloads.decode_batch(BATCH, CTX_LO, CTX_HI, seed=seed + 1, vocab=cfg["vocab_size"], spare_blocks=64)
    runner = ModelRunner.__new__(ModelRunner)
    runner.device, runner.block_size, runner.max_model_len = dev, 16, 4096  # as the decode step's runner
    kv = torch.empty(cfg["num_hidden_layers"], 2, batch.num_blocks * 16, cfg["num_key_value_heads"], cfg["head_dim"],
                     dtype=torch.bfloat16, device=dev)
    workloads.fill_kv_pool_(kv, seed=seed + 2, on_device=True)
    runner.kv_caches = [(kv[i, 0], kv[i, 1]) for i in range(kv.shape[0])]
    sched = decode_sched(cfg, batch, seed + 3)
    secs, nbytes, kname = time_layer_attention(runner, sched, cfg)
    print(json.dumps({"kernel": kname, "us_per_launch": secs * 1e6, "bytes_per_launch": nbytes,
                      "GB_s": nbytes / secs / 1e9}))
    return 0


def bench_sample(args) -> dict:
    """Sampling of a decode batch: 64 rows of Qwen3 vocabulary logits, temperature 0.8, top-k 50
    and top-p 0.9 on every row, the exponential race on Exp(1) noise -> ids."""
    import torch

    from miniserve_amd import kernels

    dev = torch.device("cuda:0")
    rows, vocab = BATCH, 151936
    copies = 8  # 8 x 78 MB of logits + noise: repeats cannot come from the Infinity Cache
    g = torch.Generator(device=dev).manual_seed(args.seed)
    logits = [torch.randn(rows, vocab, generator=g, device=dev) * 3 for _ in range(copies)]
    noise = [torch.empty(rows, vocab, device=dev).exponential_(generator=g) for _ in range(copies)]
    temps = torch.full((rows,), 0.8, device=dev)
    top_k = torch.full((rows,), 50, dtype=torch.int32, device=dev)
    top_p = torch.full((rows,), 0.9, device=dev)
    greedy = torch.zeros(rows, dtype=torch.uint8, device=dev)

    def launch(i):
        kernels.sample_ids(logits[i], temps, top_k, top_p, greedy, noise[i])

    secs = hip_time(launch, copies)
    # The logits, read once; the noise is read only at the few candidates that reach the race.
    nbytes = rows * vocab * 4
    gbs = nbytes / secs / 1e9
    log(f"sampling {rows} x {vocab}: {secs * 1e6:.1f} us/launch")
    out = line("sampling tok/s (64 rows x 151936 vocab, temperature + top-k 50 + top-p 0.9)", rows / secs, "tok/s", args,
               secs * 1e3, {"workload": "runner/sampler.py sample() on float32 logits with caller noise",
                            "rows": rows, "vocab": vocab, "temperature": 0.8, "top_k": 50, "top_p": 0.9})
    out["roofline"] = roofline("sample_chunk_kernel + sample_finish_kernel (the whole call)", "hbm", gbs, nbytes, secs)
    if not args.no_cpu_baseline:
        from oracle import sampler as osm

        torch.set_num_threads(cpu_threads())
        lc, nc = logits[0].cpu(), noise[0].cpu()
        tc, kc, pc, gc = temps.cpu(), top_k.cpu().long(), top_p.cpu(), greedy.cpu().bool()
        med, reps = cpu_time(lambda: osm.sample(lc, tc, kc, pc, gc, nc), budget_s=15.0, max_reps=20)
        out["cpu_baseline"] = cpu_fields(rows / med, "tok/s", f"the same 64 rows on the CPU oracle (the reference's "
                                         f"sort-based top-k / top-p), median of {reps}")
    return out


WORKLOADS = {"decode": bench_decode, "linear": bench_linear, "attention": bench_attention, "prefill": bench_prefill,
             "decode8b": bench_decode8b, "sample": bench_sample, "longctx": bench_long_context}


def main() -> int:
    ap = argparse.ArgumentParser()
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=20)
    ap.add_argument("--warmup", type=int, default=5)
    ap.add_argument("--seed", type=int, default=0)
    ap.add_argument("--no-cpu-baseline", action="store_true")
    ap.add_argument("--no-extra-workloads", action="store_true",
                    help="default line only: skip the chunked-prefill and 8B-shaped steps measured beside it")
    ap.add_argument("--workload", choices=sorted(WORKLOADS), default="decode")
    ap.add_argument("--kernel-only", choices=["attention", "linear", "copy", "step-linears", "gemm", "prefill-attention",
                                              "single-linear", "paged-attention"],
                    help="profiling entry point")
    args = ap.parse_args()
    if args.gpus != 1 or int(os.environ.get("WORLD_SIZE", "1")) != 1:
        print("bench.py measures one GPU only: this build has no multi-GPU path (run with --gpus 1)", file=sys.stderr)
        return 2
    if args.kernel_only:
        return kernel_only(args.kernel_only, args.seed)
    out = WORKLOADS[args.workload](args)
    if args.workload == "decode" and not args.no_extra_workloads:
        out.update(extra_workloads(args))
    print(json.dumps(out))
    return 0


def extra_workloads(args) -> dict:
    """The chunked-prefill step and the Qwen3-8B-shaped decode step, 10 timed steps each after 3
    warm-ups, and the small-batch long-context decode attention, reported beside the default line
    (the same fields as their own lines, without a CPU baseline) so that one default run records
    every workload; ~45 s of GPU time."""
    import gc

    import torch

    sub = argparse.Namespace(**{**vars(args), "steps": 10, "warmup": 3, "no_cpu_baseline": True})
    keep = ("metric", "value", "unit", "ms_per_step", "steps", "warmup", "higher_is_better", "config", "roofline",
            "roofline_gemm", "sweep")
    out = {}
    for key, fn in (("chunked_prefill", bench_prefill), ("qwen3_8b_decode", bench_decode8b),
                    ("long_context_attention", bench_long_context)):
        gc.collect()
        torch.cuda.empty_cache()
        r = fn(sub)
        out[key] = {k: r[k] for k in keep if k in r}
    return out


if __name__ == "__main__":
    sys.exit(main())
