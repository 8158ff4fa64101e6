"""Turn scheduled sequences into one forward pass and greedy next tokens (reference:
src/miniserve/runner/model_runner.py).

The runner owns the KV pool ``[layers, 2, num_blocks * block_size, kv_heads, head_dim]``
(model_runner.py:77-94, zero-filled so masked slots never hold NaN), flattens every scheduled
sequence's new tokens into one batch with per-token positions and slots (model_runner.py:162-205),
computes logits only for rows that are sampled and syncs once per step (model_runner.py:207-239).
The engine, scheduler and block manager stay with the caller: a ``ScheduledChunk`` carries what the
runner reads from the reference's ``ScheduledSeq`` (token ids, tokens already computed, tokens
scheduled now, block table) and, for a sampled request, its ``SamplingParams`` and generator.
Greedy steps sample inside the fused LM head + argmax; steps with temperature / top-k / top-p rows
compute the sampled rows' logits and run the sampling kernel (runner/sampler.py).

Pure decode steps (every sequence schedules one token) run as a captured HIP graph per batch size
(``use_graphs``): the forward, the LM head and the greedy argmax replay with one launch. The
step's ids, positions, slots and context lengths are packed (by the ``_hostprep`` extension) into
a pinned host buffer that the graph's first node uploads; the block tables sit in a second one,
uploaded before the replay only when a row changed. This is the reference's own next step
(its README's "CUDA graphs" item): its decode step is launch-bound.
"""

from __future__ import annotations

from dataclasses import dataclass
from typing import Any

import numpy as np
import torch
from torch import Tensor

try:
    from miniserve_amd import _hostprep
except ImportError as e:  # the in-tree CPython extension built with the HIP library
    raise ImportError("miniserve_amd/_hostprep is not built: run `python -m miniserve_amd.build`") from e
from miniserve_amd.attention.backends import PREFILL_TILE_SIZES, AttentionMetadata, DecodePlan, metadata_from_parts
from miniserve_amd.kernels import DEC_MAX_TOKENS
from miniserve_amd.model.qwen3 import Qwen3ForCausalLM
from miniserve_amd.runner.sampler import sample


@dataclass
class ScheduledChunk:
    token_ids: list[int]
    num_computed: int
    num_new: int
    block_table: list[int]
    params: Any = None  # the request's SamplingParams (temperature, top_k, top_p, greedy); None: greedy
    generator: torch.Generator | None = None  # a seeded request's generator (model_runner.py:_generator)

    @property
    def greedy(self) -> bool:
        return self.params is None or bool(self.params.greedy)


@dataclass
class StepInputs:
    input_ids: Tensor
    positions: Tensor
    attn: AttentionMetadata
    logits_rows: Tensor
    sample_idx: list[int]


@dataclass(frozen=True)
class _Greedy:
    temperature: float = 0.0
    top_k: int = -1
    top_p: float = 1.0
    greedy: bool = True


_GREEDY = _Greedy()


class CapturedDecode:
    """One decode step of ``batch`` sequences captured as a HIP graph with static inputs.

    Block tables are ``max_blocks`` wide (the longest context the graph accepts is
    ``max_blocks * block_size`` tokens); the attention launch shape depends only on that width.
    The per-step inputs live in two pinned host buffers: the header (ids, positions, slots as
    int64; plan rows and context lengths as int32) is uploaded every step, the block-table rows
    only on steps where one of them changed (most decode steps append no block).
    """

    def __init__(self, runner: ModelRunner, batch: int, max_blocks: int) -> None:
        dev = runner.device
        self.batch, self.max_blocks = batch, max_blocks
        b = batch
        self.host = torch.zeros(3 * b + b, dtype=torch.int64, pin_memory=True)  # ids | pos | slots | int32 pairs
        self.host_tab = torch.zeros(b * max_blocks, dtype=torch.int32, pin_memory=True)
        self.dev = torch.zeros_like(self.host, device=dev)
        self.dev_tab = torch.zeros_like(self.host_tab, device=dev)
        self.rows = torch.arange(b, dtype=torch.int64, device=dev)  # every row is sampled
        self.ids, self.pos, self.slots = self.dev[:b], self.dev[b : 2 * b], self.dev[2 * b : 3 * b]
        meta32 = self.dev[3 * b :].view(torch.int32)  # q_rows | context_lens, as int32
        # own_slots: run() checks every step (larger batches write the keys before they attend)
        plan = DecodePlan(meta32[:b], meta32[b : 2 * b], self.dev_tab.view(b, max_blocks), runner.split_context, True)
        self.meta = AttentionMetadata(self.slots, runner.block_size, plan, None)
        self.host_meta = self.host[3 * b :].view(torch.int32).numpy()
        self.host_i64 = self.host[: 3 * b].numpy()
        self.host_tables = self.host_tab.numpy()
        self.host_meta[:b] = np.arange(b, dtype=np.int32)
        self.host_meta[b : 2 * b] = 1
        self.host_i64[2 * b : 3 * b] = -1  # warm-up rows write no KV slot (kernels skip slot < 0)
        self.dev.copy_(self.host)
        self.dev_tab.copy_(self.host_tab)
        model = runner.model
        # Warm-up and capture on one stream: workspaces are kept per stream, so the warm-up
        # reserves exactly the buffers the captured kernels use.
        self.stream = stream = torch.cuda.Stream(device=dev)
        stream.wait_stream(torch.cuda.current_stream(dev))
        with torch.cuda.stream(stream), torch.inference_mode():
            for _ in range(2):
                model.greedy(self.ids, self.pos, runner.kv_caches, self.meta, self.rows)
        torch.cuda.current_stream(dev).wait_stream(stream)
        self.graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(self.graph, stream=stream), torch.inference_mode():
            # The header's upload is the graph's first node: it copies whatever the pinned buffer
            # holds when the graph runs.
            self.dev.copy_(self.host, non_blocking=True)
            self.out_ids = model.greedy(self.ids, self.pos, runner.kv_caches, self.meta, self.rows)

    def run(self, scheduled: list[ScheduledChunk], block_size: int, limit: int) -> list[int] | None:
        """Replay the step for ``scheduled``; None (nothing replayed) when it is not a pure greedy
        decode step within ``limit`` positions (whose rows own their slots, where that is needed).

        ``_hostprep.pack_decode`` writes the ids, positions and slots, the attention plan rows
        (longest context first, each keeping its own q row, as build_attention_metadata orders
        them) with their context lengths, and each plan row's block-table prefix into the pinned
        buffers. The host table buffer mirrors the device copy, so it is uploaded only when some
        row changed (most decode steps append no block)."""
        rc = _hostprep.pack_decode(scheduled, block_size, limit, self.host_i64, self.host_meta, self.host_tables,
                                   self.max_blocks, self.batch <= DEC_MAX_TOKENS)
        if rc < 0:
            return None
        if rc:
            self.dev_tab.copy_(self.host_tab, non_blocking=True)
        self.graph.replay()  # uploads the header, then the step
        return self.out_ids.tolist()  # the one device -> host sync


class ModelRunner:
    def __init__(
        self,
        model: Qwen3ForCausalLM,
        device: torch.device,
        dtype: torch.dtype = torch.bfloat16,
        block_size: int = 16,
        use_graphs: bool = False,
        max_model_len: int = 4096,
    ) -> None:
        self.model = model
        self.model_cfg = model.cfg
        self.device = device
        self.dtype = dtype
        self.block_size = block_size
        self.kv_cache: Tensor | None = None
        self.kv_caches: list[tuple[Tensor, Tensor]] = []
        self.num_blocks = 0
        self.use_graphs = use_graphs
        self.max_model_len = max_model_len
        self.graphs: dict[int, CapturedDecode] = {}

    @property
    def split_context(self) -> int:
        """The longest context decode key splits are planned for: max_model_len in whole blocks,
        the same for eager steps and captured graphs (whose tables are that wide)."""
        return -(-self.max_model_len // self.block_size) * self.block_size

    @property
    def bytes_per_block(self) -> int:
        return self.model_cfg.kv_bytes_per_token(self.dtype.itemsize) * self.block_size

    def allocate_kv_cache(self, num_blocks: int) -> None:
        c = self.model_cfg
        self.kv_cache, self.kv_caches = None, []
        self.kv_cache = torch.zeros(
            c.num_hidden_layers, 2, num_blocks * self.block_size, c.num_key_value_heads, c.head_dim,
            dtype=self.dtype, device=self.device,
        )
        self.kv_caches = [(self.kv_cache[i, 0], self.kv_cache[i, 1]) for i in range(c.num_hidden_layers)]
        self.num_blocks = num_blocks
        self.graphs = {}  # captured graphs hold the old pool's addresses

    def prepare(self, scheduled: list[ScheduledChunk]) -> StepInputs:
        """Flatten all scheduled tokens into one batch (model_runner.py:162-205, no speculation).

        ``_hostprep.pack_step`` builds the ids, positions, slots, sampled rows and the attention
        plan (build_attention_metadata's parts) in one host buffer, uploaded with one pinned,
        non-blocking copy."""
        bs = self.block_size
        data, total, sample_idx, layout, own = _hostprep.pack_step(scheduled, bs, PREFILL_TILE_SIZES, DEC_MAX_TOKENS)
        n64 = 3 * total + len(sample_idx)
        host = torch.frombuffer(data, dtype=torch.uint8) if len(data) else torch.empty(0, dtype=torch.uint8)
        dev = host.to(self.device) if self.device.type != "cuda" else host.pin_memory().to(self.device, non_blocking=True)
        i64 = dev[: 8 * n64].view(torch.int64)
        slot_mapping = i64[2 * total : 3 * total]
        return StepInputs(
            input_ids=i64[:total],
            positions=i64[total : 2 * total],
            attn=metadata_from_parts(dev[8 * n64 :].view(torch.int32), layout, slot_mapping, bs, self.split_context, own),
            logits_rows=i64[3 * total :],
            sample_idx=sample_idx,
        )

    def _graphable(self, scheduled: list[ScheduledChunk]) -> bool:
        """A pure greedy decode step: every sequence schedules its one new token, within
        max_model_len (the condition ``CapturedDecode.run`` checks again on every step)."""
        limit = self.max_model_len
        for s in scheduled:
            p, params = s.num_computed, s.params
            if s.num_new != 1 or p + 1 != len(s.token_ids) or not 0 <= p < limit or not (params is None or params.greedy):
                return False
        return True

    @torch.inference_mode()
    def forward_logits(self, inp: StepInputs) -> Tensor:
        """Logits of the sampled rows (runner/model_runner.py:214-217)."""
        return self.model.logits(inp.input_ids, inp.positions, self.kv_caches, inp.attn, inp.logits_rows)

    @torch.inference_mode()
    def forward_greedy(self, inp: StepInputs) -> Tensor:
        """Greedy ids of the sampled rows, the same as ``sample(forward_logits(inp))`` without
        materializing the logits (final norm, LM head and argmax fused)."""
        return self.model.greedy(inp.input_ids, inp.positions, self.kv_caches, inp.attn, inp.logits_rows)

    def execute(self, scheduled: list[ScheduledChunk]) -> list[list[int]]:
        """Run one step; return each scheduled sequence's new token ids (0 or 1 of them)."""
        if self.use_graphs and scheduled:
            g = self.graphs.get(len(scheduled))
            if g is None and self._graphable(scheduled):
                # positions up to max_model_len - 1 are graphable: ceil(max_model_len / block_size)
                # table entries, the last block possibly partial
                width = -(-self.max_model_len // self.block_size)
                g = self.graphs[len(scheduled)] = CapturedDecode(self, len(scheduled), width)
            # The replay needs no inference mode (its buffers are written by copies only).
            ids = g.run(scheduled, self.block_size, self.max_model_len) if g is not None else None
            if ids is not None:
                return [[t] for t in ids]
        return self._execute_eager(scheduled)

    @torch.inference_mode()
    def _execute_eager(self, scheduled: list[ScheduledChunk]) -> list[list[int]]:
        results: list[list[int]] = [[] for _ in scheduled]
        if not scheduled:
            return results
        inp = self.prepare(scheduled)
        if inp.logits_rows.numel() == 0:
            self.model(inp.input_ids, inp.positions, self.kv_caches, inp.attn)
            return results
        sampled = [scheduled[i] for i in inp.sample_idx]
        if all(s.greedy for s in sampled):
            tokens = self.forward_greedy(inp).tolist()  # the one device -> host sync
        else:  # temperature / top-k / top-p rows: logits of the sampled rows, then the sampling kernel
            logits = self.forward_logits(inp)
            params = [s.params if s.params is not None else _GREEDY for s in sampled]
            tokens = sample(logits, params, [s.generator for s in sampled]).tolist()
        for j, idx in enumerate(inp.sample_idx):
            results[idx] = [tokens[j]]
        return results
