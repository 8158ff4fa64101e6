"""GPU parity of the wide decode linear (gemv_wide.hip), which msa_int8_linear takes for up to 64 tokens
over weights of 12 MB and more (and msa_int8_linear_add_rmsnorm with it, in one launch or merging
split-K partials), against the CPU oracle on the same seeded inputs; and of the large-weight decode
layers against the general layer loop.

Same operands and rounding points as the oracle's bf16 product, float32 accumulation in another
order: within rel-L2 2e-3 of the oracle and within one bf16 rounding (4e-3) of float64, as the other
decode linears. Shapes take every unit width (1, 2, 3, 6 tiles) and token-tile count, ragged last
units, K whose chunks do not deal evenly to the eight wavefronts, 1 and 64 tokens. The kernel is taken
where it is the faster one: shapes to either side of those lines, on whatever serves them."""

from __future__ import annotations

import pytest
import torch
from helpers import rel_l2
from model_helpers import copy_pool_to_oracle, oracle_step, pair

from miniserve_amd import _native, kernels, workloads
from miniserve_amd.attention import backends
from miniserve_amd.model import qwen3
from miniserve_amd.quant.int8 import quantize_int8_
from miniserve_amd.runner.model_runner import ModelRunner, ScheduledChunk
from oracle import int8 as oi
from oracle import layers as ol

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")


def _bf16(shape, seed, std=1.0):
    return (torch.randn(shape, generator=torch.Generator().manual_seed(seed)) * std).to(torch.bfloat16)


WIDE_SHAPES = [  # (m, n, k)
    (1, 4090, 4160),  # one tile per unit, ragged n, 65 chunks
    (16, 3072, 4160),
    (5, 6150, 3136),  # two tiles, 49 chunks
    (13, 12290, 1088),  # 769 tiles in twos, 17 chunks
    (3, 12280, 1088),  # three tiles
    (13, 12280, 1088),
    (17, 4096, 3136),
    (32, 6144, 3136),
    (20, 12280, 1088),
    (32, 24560, 576),  # six tiles, 9 chunks
    (33, 4096, 3136),
    (47, 6150, 3136),
    (48, 12290, 1088),
    (49, 4090, 3136),
    (64, 6144, 3136),
    (63, 12290, 1088),
    (40, 12280, 1088),  # three tiles
    (60, 12280, 1088),
    (32, 2048, 8256),  # split K, merged by the epilogue kernel
    (64, 1600, 8256),
    (40, 2048, 6208),
]


@pytest.mark.parametrize("m,n,k", WIDE_SHAPES)
def test_wide_linear(m, n, k):
    assert n * k >= kernels.WIDE_MIN_WEIGHTS
    q, s = oi.quantize_int8(_bf16((n, k), seed=n + k, std=0.02))
    x, r = _bf16((m, k), seed=m), _bf16((m, n), seed=m + 1)
    xd, qd, sd, rd = (t.to(DEV) for t in (x, q, s, r))
    y = kernels.int8_linear(xd, qd, sd)
    assert torch.equal(y, kernels.int8_linear(xd, qd, sd))
    exact = x.double() @ oi.dequantize(q, s, torch.bfloat16).double().T
    assert rel_l2(y.cpu(), oi.int8_linear(x, q, s)) < 2e-3
    assert rel_l2(y.cpu(), exact) < 4e-3
    # without a workspace: one launch, K never split; strided x and y rows
    xs = torch.zeros(m, k + 64, dtype=torch.bfloat16, device=DEV)
    xs[:, :k] = xd
    y2 = torch.zeros(m, n + 8, dtype=torch.bfloat16, device=DEV)
    _native.call("msa_int8_linear", kernels._ptr(xs), m, k, k + 64, kernels._ptr(qd), kernels._ptr(sd), n,
                 kernels._ptr(y2), n + 8, 0, None, 0, None, 0, kernels._stream(y2))
    assert rel_l2(y2[:, :n].cpu(), exact) < 4e-3 and not y2[:, n:].any()
    # residual added to the rounded product, in place
    acc = rd.clone()
    kernels.int8_linear(xd, qd, sd, kernels.EPI_RESIDUAL, residual=acc, out=acc)
    assert torch.equal(acc, (rd.float() + y.float()).to(torch.bfloat16))
    # silu(gate) * up of the two halves
    gate, up = exact.to(torch.bfloat16).chunk(2, dim=-1)
    act = kernels.int8_linear(xd, qd, sd, kernels.EPI_SILU_MUL)
    assert rel_l2(act.cpu(), torch.nn.functional.silu(gate) * up) < 8e-3


@pytest.mark.parametrize("m,n,k", [  # to either side of the rules that choose the kernel for large weights
    (16, 1024, 12352), (16, 2560, 4992), (20, 448, 28160), (9, 4096, 3072), (24, 6144, 2048), (8, 8192, 1536),
    (70, 1024, 12288), (70, 2048, 6144), (100, 8192, 2048), (127, 4096, 4096), (65, 8448, 1536),
])
def test_large_weight_routes(m, n, k):
    """Every epilogue, whichever kernel it takes (they need not agree): within one bf16 rounding of float64
    (two with the residual's own sum, three with silu(gate) * up)."""
    q, s = oi.quantize_int8(_bf16((n, k), seed=n + k, std=0.02))
    x, r, w = _bf16((m, k), seed=m), _bf16((m, n), seed=m + 1), _bf16((n,), seed=3, std=0.1) + 1
    xd, qd, sd, rd = (t.to(DEV) for t in (x, q, s, r))
    exact = x.double() @ oi.dequantize(q, s, torch.bfloat16).double().T
    assert rel_l2(kernels.int8_linear(xd, qd, sd).cpu(), exact) < 4e-3
    assert rel_l2(kernels.int8_linear(xd, qd, sd, kernels.EPI_RESIDUAL, residual=rd).cpu(), exact + r.double()) < 8e-3
    gate, up = exact.chunk(2, dim=-1)
    act = kernels.int8_linear(xd, qd, sd, kernels.EPI_SILU_MUL).cpu()
    assert rel_l2(act, gate * torch.sigmoid(gate) * up) < 1.2e-2
    res = rd.clone()
    out = kernels.int8_linear_add_rmsnorm(xd, qd, sd, res, w.to(DEV), 1e-6)
    assert rel_l2(res.cpu(), exact + r.double()) < 8e-3
    assert rel_l2(out.cpu(), ol.rms_norm(res.cpu(), w, 1e-6)) < 2e-3


@pytest.mark.parametrize("m,n,k", [(1, 4096, 4160), (16, 2048, 8256), (17, 4096, 3136), (40, 2048, 8256), (64, 2568, 4992)])
def test_wide_linear_add_rmsnorm(m, n, k):
    q, s = oi.quantize_int8(_bf16((n, k), seed=n + k, std=0.02))
    x, r, w = _bf16((m, k), seed=m), _bf16((m, n), seed=m + 1), _bf16((n,), seed=3, std=0.1) + 1
    res = r.to(DEV)
    out = kernels.int8_linear_add_rmsnorm(x.to(DEV), q.to(DEV), s.to(DEV), res, w.to(DEV), 1e-6)
    ref = r + oi.int8_linear(x, q, s)
    assert rel_l2(res.cpu(), ref) < 2e-3
    assert rel_l2(out.cpu(), ol.rms_norm(res.cpu(), w, 1e-6)) < 2e-3  # of its own sum: the order of squares


@pytest.mark.parametrize("batch", [1, 16, 17, 64, 70])
def test_wide_decode_layers_match_the_layer_loop(batch, monkeypatch):
    """The large-weight decode layers against the general loop on the same model and pool: the same
    values but for the orders of float32 sums, amplified by bf16 roundings over two layers (each
    route measures about 1.4e-2 from float64 on this shape)."""
    cfg = {**workloads.QWEN3_8B, "num_hidden_layers": 2, "vocab_size": 512, "tie_word_embeddings": True}
    model = workloads.build_model(cfg, workloads.random_weights(cfg, 5, norm_jitter=0.1, device="cuda"), DEV, 256)
    quantize_int8_(model)
    runner = ModelRunner(model, DEV, max_model_len=256)
    ctx = [3 + (37 * i) % 200 for i in range(batch)]
    blocks = [-(-c // 16) for c in ctx]
    perm = torch.randperm(sum(blocks), generator=torch.Generator().manual_seed(1)).tolist()
    tables, off = [], 0
    for b in blocks:
        tables.append(perm[off : off + b])
        off += b
    sched = [ScheduledChunk([(7 * i + j) % 512 for j in range(c)], c - 1, 1, t) for i, (c, t) in enumerate(zip(ctx, tables))]
    got = []
    for wide in (True, False):
        if not wide:
            monkeypatch.setattr(type(model), "_wide_decode_ok", lambda self, tokens, meta: False)
        runner.allocate_kv_cache(sum(blocks))
        workloads.fill_kv_pool_(runner.kv_cache, 9, on_device=True)
        inp = runner.prepare(sched)
        assert model._wide_decode_ok(batch, inp.attn) is wide
        with torch.inference_mode():
            got.append((model(inp.input_ids, inp.positions, runner.kv_caches, inp.attn), runner.kv_cache.clone()))
    assert rel_l2(got[0][0].cpu(), got[1][0].cpu()) < 2e-2
    assert rel_l2(got[0][1].cpu(), got[1][1].cpu()) < 5e-3


@pytest.mark.parametrize("m,n,k", [(5, 6150, 3136), (20, 12280, 1088), (64, 6144, 3136), (64, 1600, 8256)])
def test_wide_non_finite_rows(m, n, k):
    """Infinities and NaN in single rows: those rows as a float32 product has them (0 * inf is NaN), the
    others bit for bit what they are without."""
    q, s = oi.quantize_int8(_bf16((n, k), seed=n + k, std=0.02))
    x = _bf16((m, k), seed=m)
    clean = kernels.int8_linear(x.to(DEV), q.to(DEV), s.to(DEV)).cpu()
    x[0, k - 1], x[2, 5], x[m - 1, 0] = float("inf"), float("nan"), float("-inf")
    x[3, 7], x[3, 70] = float("inf"), float("-inf")
    y = kernels.int8_linear(x.to(DEV), q.to(DEV), s.to(DEV)).cpu()
    bad = sorted({0, 2, 3, m - 1})
    want = (x[bad].float() @ oi.dequantize(q, s, torch.bfloat16).float().T).to(torch.bfloat16)
    assert not want.isfinite().any() and (want == float("inf")).any() and want.isnan().any()
    assert torch.equal(y[bad].nan_to_num(7.0), want.nan_to_num(7.0)) and torch.equal(y[bad].isnan(), want.isnan())
    keep = [i for i in range(m) if i not in bad]
    assert torch.equal(y[keep], clean[keep])


# One layer whose linears all reach WIDE_MIN_WEIGHTS and whose down projection is past the token-split kernels.
LARGE = {**workloads.QWEN3_8B, "num_hidden_layers": 1, "intermediate_size": 4608, "vocab_size": 512,
         "tie_word_embeddings": True}


@pytest.mark.parametrize("batch", [3, 20])
@pytest.mark.parametrize("hidden,heads,kv_heads", [(3584, 32, 32), (3584, 32, 16), (4096, 32, 4), (3584, 32, 8)])
def test_wide_decode_layers_of_other_shapes(hidden, heads, kv_heads, batch, monkeypatch):
    """Every group size, and hidden sizes that the decode kernel does not take (3584: the norms then run
    with the o and down projections for few tokens too), against the general loop at the bars above."""
    cfg = {**LARGE, "hidden_size": hidden, "num_attention_heads": heads, "num_key_value_heads": kv_heads}
    runner, sched = _decode_step(cfg, batch)
    inp = runner.prepare(sched)
    assert not runner.model._token_split_ok(batch) and runner.model._wide_decode_ok(batch, inp.attn)
    got = _forward(runner, inp, 4 * batch)
    monkeypatch.setattr(type(runner.model), "_wide_decode_ok", lambda self, tokens, meta: False)
    want = _forward(runner, inp, 4 * batch)
    assert rel_l2(got[0], want[0]) < 2e-2 and rel_l2(got[1], want[1]) < 5e-3
    slots = inp.attn.slot_mapping.cpu()
    assert rel_l2(got[1][0, :, slots], want[1][0, :, slots]) < 1e-2


def _decode_step(cfg, batch, blocks_each=4, seed=5):
    """(runner, scheduled decode rows of 3 to 60 tokens): a seeded int8 model, each sequence in blocks of
    its own."""
    model = workloads.build_model(cfg, workloads.random_weights(cfg, seed, norm_jitter=0.1, device="cuda"), DEV, 256)
    quantize_int8_(model)
    runner = ModelRunner(model, DEV, max_model_len=256)
    ctx = [3 + (37 * i) % (16 * blocks_each - 6) for i in range(batch)]
    perm = torch.randperm(batch * blocks_each, generator=torch.Generator().manual_seed(1)).tolist()
    return runner, [ScheduledChunk([(7 * i + j) % cfg["vocab_size"] for j in range(c)], c - 1, 1,
                                   perm[blocks_each * i : blocks_each * (i + 1)]) for i, c in enumerate(ctx)]


def _forward(runner, inp, blocks, positions=None):
    """(hidden states, KV pool) of one forward over a freshly filled pool."""
    runner.allocate_kv_cache(blocks)
    workloads.fill_kv_pool_(runner.kv_cache, 9, on_device=True)
    with torch.inference_mode():
        out = runner.model(inp.input_ids, inp.positions if positions is None else positions, runner.kv_caches, inp.attn)
    return out.cpu(), runner.kv_cache.cpu()


@pytest.mark.parametrize("batch", [3, 20])
def test_wide_decode_layers_rotate_by_the_given_positions(batch, monkeypatch):
    """forward(input_ids, positions, ...) with positions other than the contexts' last ones (a shifted
    window, say): the large-weight decode layers rotate by them as the general loop does, and write
    the keys so rotated (bars as in the test above; another rotation is off by 0.1 and more)."""
    runner, sched = _decode_step(LARGE, batch)
    inp = runner.prepare(sched)
    positions = (inp.positions * 3 + 41) % 256
    assert not runner.model._token_split_ok(batch) and runner.model._wide_decode_ok(batch, inp.attn)
    own, got = _forward(runner, inp, 4 * batch), _forward(runner, inp, 4 * batch, positions)
    other = _forward(runner, inp, 4 * batch, positions.int().cpu())  # as indexing takes them
    assert torch.equal(other[0], got[0]) and torch.equal(other[1], got[1])
    monkeypatch.setattr(type(runner.model), "_wide_decode_ok", lambda self, tokens, meta: False)
    want = _forward(runner, inp, 4 * batch, positions)
    assert rel_l2(got[0], want[0]) < 2e-2 and rel_l2(got[1], want[1]) < 5e-3
    slots = inp.attn.slot_mapping.cpu()
    assert rel_l2(got[1][0, 0, slots], want[1][0, 0, slots]) < 1e-2
    assert rel_l2(own[1][0, 0, slots], want[1][0, 0, slots]) > 0.1


def _twice(sched):
    """The batch with its first sequence in it again, one token further (a verify as single rows, say)."""
    s = sched[0]
    return [*sched, ScheduledChunk([*s.token_ids, 11], s.num_computed + 1, 1, s.block_table)]


def test_large_model_rows_that_share_a_slot_take_the_layer_loop(monkeypatch):
    """Two rows of one sequence: the later attends to the key that the earlier writes in this step. The
    large-weight decode layers write keys inside the attention launch, so such a batch, and one whose
    slots the plan's builder did not make, takes the general loop, which writes every key first."""
    runner, sched = _decode_step(LARGE, 3)
    inp = runner.prepare(sched)
    seqs = [backends.SeqChunk(i, 1, s.num_computed, s.block_table) for i, s in enumerate(sched)]
    assert runner.model._wide_decode_ok(3, inp.attn)
    assert not runner.model._wide_decode_ok(3, backends.build_attention_metadata(seqs, inp.attn.slot_mapping, 16))
    inp = runner.prepare(_twice(sched))
    assert not runner.model._wide_decode_ok(4, inp.attn)
    got = _forward(runner, inp, 12)
    monkeypatch.setattr(type(runner.model), "_wide_decode_ok", lambda self, tokens, meta: False)
    want = _forward(runner, inp, 12)
    assert torch.equal(got[0], want[0]) and torch.equal(got[1], want[1])


def test_small_model_rows_that_share_a_slot(monkeypatch):
    """The same batch on the token-split pipeline, eager and where a graph of its size is captured: keys
    written before any row attends, logits as the oracle's (which writes, then attends)."""
    cfg = {**workloads.QWEN3_0_6B, "num_hidden_layers": 1, "vocab_size": 1024}
    runner, ocfg, ow, okv, tables = pair(cfg, seed=3, max_positions=256, num_blocks=16)
    workloads.fill_kv_pool_(runner.kv_cache, seed=4)
    copy_pool_to_oracle(runner, okv)
    runner.use_graphs, runner.max_model_len = True, 256
    ctx = [20, 33, 7]
    sched = [ScheduledChunk([(5 * i + j) % 1024 for j in range(c)], c - 1, 1, list(range(4 * i, 4 * i + 4)))
             for i, c in enumerate(ctx)]
    before = runner.kv_cache.clone()
    runner.execute([*sched, ScheduledChunk([1, 2], 1, 1, [13])])  # captures a graph of four rows
    assert list(runner.graphs) == [4]
    runner.kv_cache.copy_(before)
    shared = _twice(sched)
    logits, ids = oracle_step(ocfg, ow, okv, tables, shared)

    def never(*args, **kwargs):
        raise AssertionError("attention that writes the keys itself")

    monkeypatch.setattr(qwen3, "attend_decode_qkv", never)
    assert rel_l2(runner.forward_logits(runner.prepare(shared)).cpu(), logits) < 1e-2
    runner.kv_cache.copy_(before)
    assert [r[0] for r in runner.execute(shared)] == runner.forward_greedy(runner.prepare(shared)).tolist()
    slots = runner.prepare(shared).attn.slot_mapping.cpu()
    assert rel_l2(runner.kv_caches[0][0].cpu()[slots], okv[0][0][slots]) < 1e-2


@pytest.mark.parametrize("m,n,k,fused", [
    (27, 4096, 4096, False),  # needs nothing
    (27, 4096, 4096, True),  # partials where there is room for them
    (96, 4096, 4096, False),
    (96, 4096, 4096, True),
])
def test_capture_without_a_reserved_workspace(m, n, k, fused, monkeypatch):
    """Linears whose splits are a gain and no need are captured on a stream that holds no workspace, and then
    run unsplit: replayed three times with eager work between, within one bf16 rounding of float64."""
    monkeypatch.setattr(kernels, "workspaces", kernels._Workspaces())
    q, s = oi.quantize_int8(_bf16((n, k), seed=n + k, std=0.02))
    x, r = _bf16((m, k), seed=m), _bf16((m, n), seed=m + 1)
    xd, qd, sd, rd, res = x.to(DEV), q.to(DEV), s.to(DEV), r.to(DEV), torch.empty(m, n, dtype=torch.bfloat16, device=DEV)
    w = torch.ones(n, dtype=torch.bfloat16, device=DEV)

    def run():
        if not fused:
            return kernels.int8_linear(xd, qd, sd)
        res.copy_(rd)
        kernels.int8_linear_add_rmsnorm(xd, qd, sd, res, w, 1e-6)
        return res

    eager = run().clone()  # (also loads the kernels)
    exact = x.double() @ oi.dequantize(q, s, torch.bfloat16).double().T + (r.double() if fused else 0.0)
    stream, graph = torch.cuda.Stream(), torch.cuda.CUDAGraph()
    torch.cuda.synchronize()
    with torch.cuda.graph(graph, stream=stream):
        out = run()
    for _ in range(3):
        graph.replay()
        torch.cuda.synchronize()
        assert rel_l2(out.cpu(), exact) < 4e-3
        xd.mul_(1.0)
    assert rel_l2(out.cpu(), eager.cpu()) < 4e-3


def test_capture_still_wants_the_needed_workspace(monkeypatch):
    """Splits without which most of the chip is idle are still to be reserved: refused during a capture."""
    q, s = oi.quantize_int8(_bf16((4096, 4096), seed=1, std=0.02))
    x, qd, sd = _bf16((256, 4096), seed=2).to(DEV), q.to(DEV), s.to(DEV)
    monkeypatch.setattr(kernels, "workspaces", kernels._Workspaces())
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: True)
    with pytest.raises(RuntimeError, match="must be reserved before graph capture"):
        kernels.int8_linear(x, qd, sd)
    kernels.workspaces._bufs["linear", 0, torch.cuda.current_stream().cuda_stream] = torch.empty(16 << 20, dtype=torch.uint8, device=DEV)
    kernels.int8_linear(x, qd, sd)


@pytest.mark.parametrize("t,hidden", [(1, 8), (3, 4096), (128, 8200)])
def test_embed_rope_rows(t, hidden):
    """The embedding and rotary gathers of the large-model decode step, bit for bit: one piece to several
    pieces per thread, first and last entries, positions counted from the end."""
    g = torch.Generator().manual_seed(hidden)
    weight, cos, sin = _bf16((50, hidden), seed=t).to(DEV), torch.randn(70, 128, generator=g).to(DEV), torch.randn(70, 128, generator=g).to(DEV)
    ids, pos = torch.randint(0, 50, (t,), generator=g), torch.randint(-70, 70, (t,), generator=g)
    ids[0], pos[0], ids[-1], pos[-1] = 0, -70, 49, 69
    ids, pos = ids.to(DEV), pos.to(DEV)
    x, c, s = kernels.embed_rope_rows(ids, pos, weight, cos, sin)
    assert torch.equal(x, weight[ids]) and torch.equal(c, cos[pos]) and torch.equal(s, sin[pos])
    with pytest.raises(RuntimeError, match="ids and positions"):
        kernels.embed_rope_rows(ids, pos[:-1] if t > 1 else torch.cat([pos, pos]), weight, cos, sin)
