"""Paged attention over a slot pool, read in place by HIP kernels (reference:
src/miniserve/attention/backends.py).

Per layer the pool is ``[num_slots, kv_heads, head_dim]`` with slot = block * block_size + offset.
Each step (backends.py:145-197): write the new tokens' keys/values at ``slot_mapping``, then every
new token attends to positions 0..its own through its sequence's block table.

What differs from the reference is the plan, not the result: instead of gathering each sequence's
keys into contiguous tensors and padding groups for SDPA, ``build_attention_metadata`` prepares
int32 block tables and per-sequence lengths (one pinned, non-blocking upload per step) and the
kernels read the blocks where they lie:
  * sequences with one new token (decodes) -> split-K decode kernel;
  * sequences with more (prefill chunks, fresh or after cached keys, speculative verifies) ->
    the flash-style MFMA prefill kernel.
The metadata is built once per step and shared by all layers (backends.py:19-20).
"""

from __future__ import annotations

from dataclasses import dataclass, field

import numpy as np
import torch
from torch import Tensor

try:
    from miniserve_amd import _hostprep
except ImportError as e:  # the in-tree CPython extension built with the HIP library
    raise ImportError("miniserve_amd/_hostprep is not built: run `python -m miniserve_amd.build`") from e
from miniserve_amd import kernels
from miniserve_amd.utils import upload_int32

SHORT_QUERY = 8  # the reference's batched-path threshold (backends.py:32); kept for callers
MAX_GATHER_TOKENS = 16384  # the reference's gather cap (backends.py:33); nothing is gathered here
PREFILL_TILE = {1: 64, 2: 32, 4: 16}  # query tokens per prefill work item, by H / KVH
# Tiles of twice the tokens (32-query wavefronts) when they give at least this many workgroups, three
# for every two CUs: each key and value read from LDS then serves twice the queries (2000 tokens
# after 6000 at 32 / 8 heads, 504 workgroups: 376 -> 272 us; 2 x 2048 fresh at 16 / 8 heads, 512:
# 77 -> 56). With fewer, the longer chains of the larger tiles cost more than they save (1984 fresh
# tokens at 16 / 8 heads, 248: 38 -> 42; 500 at 32 / 8, 128: 12.5 -> 16.3), and where the tokens do not
# fill them they only double the padding (64 x 4 tokens: 58 -> 65).
PREFILL_WIDE_MIN_WORKGROUPS = 384
PREFILL_TILE_SIZES = tuple(sorted({f * t for t in PREFILL_TILE.values() for f in (1, 2)}))  # every plan's work lists


@dataclass
class SeqChunk:
    """What attention needs to know about one scheduled sequence (backends.py:36-47)."""

    flat_start: int
    num_new: int
    num_cached: int
    block_table: list[int]

    @property
    def context_len(self) -> int:
        return self.num_cached + self.num_new


@dataclass
class DecodePlan:
    q_rows: Tensor  # [B] int32 flat-batch row of each sequence's query
    context_lens: Tensor  # [B] int32
    block_tables: Tensor  # [B, max_blocks] int32, padded with block 0
    split_context: int = 0  # longest context the key splits are planned for (0: the table width)
    # Whether the slot of each row's new token is its table's slot of its last position and no other position
    # of any row's context. True: known from the packing that made the slots; False: known from the
    # tables not to be (the same sequence twice, say); None: slots made elsewhere. Attention that
    # writes the new keys in the launch that reads the contexts would race where this fails.
    own_slots: bool | None = None

    @property
    def num_seqs(self) -> int:
        return int(self.q_rows.numel())


@dataclass
class PrefillPlan:
    seq_info: Tensor  # [S, 3] int32: flat start, num_new, num_cached
    block_tables: Tensor  # [S, max_blocks] int32
    work: dict[int, Tensor] = field(default_factory=dict)  # tile tokens -> [W, 2] int32


@dataclass
class AttentionMetadata:
    slot_mapping: Tensor  # [T] int64 slot where each new token's K/V is written
    block_size: int
    decode: DecodePlan | None
    prefill: PrefillPlan | None


def context_slots(block_tables: Tensor, length: int, block_size: int) -> Tensor:
    """Slot of positions 0..length-1 through a block table (backends.py:74-77)."""
    pos = torch.arange(length, device=block_tables.device)
    return block_tables[..., pos // block_size] * block_size + pos % block_size


def _cdiv(a: int, b: int) -> int:
    return -(-a // b)


def _padded_tables(chunks: list[SeqChunk], block_size: int) -> np.ndarray:
    """[len(chunks), max blocks] int32: each chunk's first ceil(context / block_size) table
    entries, padded with block 0 (one conversion for the whole batch)."""
    needs = [_cdiv(c.context_len, block_size) for c in chunks]
    nb = max(needs)
    rows = []
    for c, need in zip(chunks, needs, strict=True):
        tab = c.block_table
        if len(tab) < need:
            raise RuntimeError(f"block table of {len(tab)} blocks is shorter than context {c.context_len}")
        rows.append(tab[:need] if need == nb else [*tab[:need], *([0] * (nb - need))])
    return np.array(rows, dtype=np.int32).reshape(len(chunks), nb)


def _prefill_work(pre: list[SeqChunk], tile: int) -> np.ndarray:
    """[W, 2] int32 (sequence, first new token) of every ``tile``-token query tile, the tiles with
    the most keys (cached + causal) first, ties in sequence then token order."""
    n = np.array([c.num_new for c in pre], dtype=np.int64)
    cached = np.array([c.num_cached for c in pre], dtype=np.int64)
    counts = -(-n // tile)
    seq = np.repeat(np.arange(len(pre), dtype=np.int64), counts)
    t0 = (np.arange(int(counts.sum()), dtype=np.int64) - np.repeat(np.cumsum(counts) - counts, counts)) * tile
    keys = cached[seq] + np.minimum(t0 + tile, n[seq])
    order = np.argsort(-keys, kind="stable")
    return np.stack([seq[order], t0[order]], axis=1).astype(np.int32)


def build_attention_metadata(
    chunks: list[SeqChunk], slot_mapping: Tensor, block_size: int, split_context: int = 0
) -> AttentionMetadata:
    """Plan one step's attention (backends.py:80-98): one int32 upload holds every table.
    ``split_context`` (optional) is the longest context the caller plans for -- the runner passes
    its max_model_len, so eager steps split decode keys as its captured graphs do."""
    if block_size != 16:
        raise RuntimeError("the HIP attention kernels use 16-token blocks")
    device = slot_mapping.device
    # Longest work first: workgroups are dispatched in grid order, so a long sequence (or a late
    # causal tile with many keys) queued last would run alone at the end. Each decode sequence
    # carries its own output row and each prefill work item its own sequence and tile, so the
    # order changes no result.
    dec = sorted((c for c in chunks if c.num_new == 1), key=lambda c: -c.context_len)
    pre = [c for c in chunks if c.num_new > 1]
    parts: list[np.ndarray] = []
    layout: list[tuple[str, tuple[int, ...]]] = []

    def add(name: str, arr: np.ndarray) -> None:
        parts.append(np.ascontiguousarray(arr, dtype=np.int32).ravel())
        layout.append((name, arr.shape))

    own_slots = None  # the slots are the caller's, on the device
    if dec:
        ctx, tables = np.array([c.context_len for c in dec], dtype=np.int32), _padded_tables(dec, block_size)
        if not _hostprep.rows_own_slots(tables, ctx, block_size):
            own_slots = False
        add("d_rows", np.array([c.flat_start for c in dec], dtype=np.int32))
        add("d_ctx", ctx)
        add("d_tables", tables)
    if pre:
        add("p_info", np.array([[c.flat_start, c.num_new, c.num_cached] for c in pre], dtype=np.int32))
        add("p_tables", _padded_tables(pre, block_size))
        for tile in PREFILL_TILE_SIZES:
            add(f"p_work{tile}", _prefill_work(pre, tile))

    flat = upload_int32(np.concatenate(parts), device) if parts else None
    return metadata_from_parts(flat, layout, slot_mapping, block_size, split_context, own_slots)


def metadata_from_parts(
    flat: Tensor | None, layout: list[tuple[str, tuple[int, ...]]], slot_mapping: Tensor, block_size: int,
    split_context: int = 0, own_slots: bool | None = None,
) -> AttentionMetadata:
    """The plan from its uploaded int32 parts: ``flat`` holds the parts named in ``layout``
    ((name, shape) pairs) back to back -- d_rows, d_ctx, d_tables for the decode sequences, p_info,
    p_tables and p_work<tile> for the prefill ones, each group present only when it has rows."""
    views: dict[str, Tensor] = {}
    off = flat.storage_offset() if flat is not None else 0
    for name, shape in layout:  # (one view each: a slice and its reshape would be two)
        two = len(shape) == 2
        views[name] = flat.as_strided(shape, (shape[1], 1) if two else (1,), off)
        off += shape[0] * shape[1] if two else shape[0]
    decode = (
        DecodePlan(views["d_rows"], views["d_ctx"], views["d_tables"], split_context, own_slots)
        if "d_rows" in views
        else None
    )
    prefill = (
        PrefillPlan(views["p_info"], views["p_tables"], {t: views[f"p_work{t}"] for t in PREFILL_TILE_SIZES})
        if "p_info" in views
        else None
    )
    return AttentionMetadata(slot_mapping, block_size, decode, prefill)


_SIDE_STREAMS: dict[int, tuple[torch.cuda.Stream, torch.cuda.Event, torch.cuda.Event]] = {}


def _side_stream(device: torch.device) -> tuple[torch.cuda.Stream, torch.cuda.Event, torch.cuda.Event]:
    """A second stream per device (default priority) for the decode rows of a mixed batch, with
    two reusable events: the fork (side waits for the caller's stream) and the join (the caller's
    stream waits for side). A wait orders against the event's latest record when the wait is
    enqueued, so re-recording them on later calls is safe."""
    idx = device.index if device.index is not None else torch.cuda.current_device()
    st = _SIDE_STREAMS.get(idx)
    if st is None:
        st = _SIDE_STREAMS[idx] = (torch.cuda.Stream(device=idx), torch.cuda.Event(), torch.cuda.Event())
    return st


def prefill_takes_wide(plan: PrefillPlan, tile: int, kv_heads: int) -> bool:
    """Whether a prefill plan runs on tiles of 2 x ``tile`` tokens: enough of them, and well filled
    (at most three for every four of the small ones)."""
    work = plan.work.get(2 * tile)
    return (work is not None and work.shape[0] * kv_heads >= PREFILL_WIDE_MIN_WORKGROUPS
            and 4 * work.shape[0] <= 3 * plan.work[tile].shape[0])


def attend(q: Tensor, k_cache: Tensor, v_cache: Tensor, meta: AttentionMetadata, scale: float) -> Tensor:
    """Attention of every new token over its cached context (the caches already hold this
    step's keys and values). q [T, H, D] -> [T, H, D].

    In a mixed batch the decode rows (HBM-bound) run on a second stream next to the prefill rows
    (MFMA-bound), in four-wavefront workgroups that fit on a CU beside a prefill workgroup; the two
    write disjoint rows of the output, and the caller's stream waits for both. The wide prefill
    tiles' wavefronts leave no registers for a decode workgroup, so mixed batches keep the small ones."""
    out = torch.empty_like(q)
    heads, kv_heads = q.shape[1], k_cache.shape[1]
    side = cur = join = None
    if meta.decode is not None and meta.prefill is not None and q.is_cuda:
        cur = torch.cuda.current_stream(q.device)
        side, fork, join = _side_stream(q.device)
        fork.record(cur)
        side.wait_event(fork)
    if meta.decode is not None:
        d = meta.decode
        ptok, parts = kernels.decode_plan(d.num_seqs, kv_heads, d.block_tables.shape[1], heads // kv_heads,
                                      d.split_context)
        kernels.paged_attention_decode(
            q, k_cache, v_cache, d.block_tables, d.context_lens, d.q_rows, ptok, parts, scale, out, meta.block_size,
            narrow=side is not None, stream=side,
        )
    if meta.prefill is not None:
        p = meta.prefill
        group = heads // kv_heads
        tile = PREFILL_TILE.get(group)
        if tile is None:
            raise RuntimeError(f"prefill attention supports H/KVH in 1, 2, 4 (got {group})")
        work = p.work[tile]
        wide = (side is None and 3 * work.shape[0] * kv_heads >= 4 * PREFILL_WIDE_MIN_WORKGROUPS
                and prefill_takes_wide(p, tile, kv_heads))  # (beside decode rows: see above)
        if wide:
            work = p.work[2 * tile]
        kernels.paged_attention_prefill(q, k_cache, v_cache, p.block_tables, p.seq_info, work, scale, out,
                                        meta.block_size, wide)
    if side is not None:
        join.record(side)
        cur.wait_event(join)
    return out


def attend_decode_qkv(
    qkv: Tensor,
    heads: int,
    q_norm_w: Tensor,
    k_norm_w: Tensor,
    qk_eps: float,
    cos_table: Tensor,
    sin_table: Tensor,
    k_cache: Tensor,
    v_cache: Tensor,
    meta: AttentionMetadata,
    scale: float,
    rope_rows: bool = False,
) -> Tensor:
    """A pure-decode step's attention from the qkv projection rows (model/qwen3.py:94-99): per-head
    q/k RMSNorm, RoPE at each sequence's new position (context length - 1, or with ``rope_rows`` by
    the row of cos_table / sin_table [T, D] of each row of qkv), the new keys and values written into
    the caches at slot_mapping (negative slots are skipped) and attention, in one kernel. The rows have
    to own their slots (DecodePlan.own_slots): keys are written in the launch that reads the contexts.
    qkv [T, (H + 2 KVH) * D] -> [T, H, D]."""
    if meta.decode is None or meta.prefill is not None:
        raise RuntimeError("attend_decode_qkv serves batches of decode rows only")
    d = meta.decode
    kv_heads, dim = k_cache.shape[1], k_cache.shape[2]
    out = torch.empty(qkv.shape[0], heads, dim, dtype=qkv.dtype, device=qkv.device)
    ptok, parts = kernels.decode_plan(d.num_seqs, kv_heads, d.block_tables.shape[1], heads // kv_heads,
                                      d.split_context)
    kernels.paged_attention_decode_qkv(
        qkv, heads, q_norm_w, k_norm_w, qk_eps, cos_table, sin_table, meta.slot_mapping, k_cache, v_cache, d.block_tables,
        d.context_lens, d.q_rows, ptok, parts, scale, out, meta.block_size, rope_rows,
    )
    return out


def paged_attention(
    q: Tensor,
    k: Tensor,
    v: Tensor,
    k_cache: Tensor,
    v_cache: Tensor,
    meta: AttentionMetadata,
    scale: float,
) -> Tensor:
    """Write this step's keys and values into the cache, then attend through it (backends.py:145-197).

    q: [T, heads, dim]; k, v: [T, kv_heads, dim]; caches: [slots, kv_heads, dim]. Returns [T, heads, dim].
    """
    kernels.reshape_and_cache(k, v, k_cache, v_cache, meta.slot_mapping)
    return attend(q, k_cache, v_cache, meta, scale)
