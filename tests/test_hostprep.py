"""The native packing of a captured decode step's inputs (``miniserve_amd/_hostprep``) against a
Python statement of the same layout: ids / positions / slots, plan rows longest context first (ties
in batch order), context lengths, block-table prefixes per plan row, and the upload flag."""

from __future__ import annotations

import random
from dataclasses import dataclass

import numpy as np
import pytest

from miniserve_amd import _hostprep


@dataclass
class Chunk:
    token_ids: list
    num_computed: int
    num_new: int
    block_table: list
    params: object = None


@dataclass
class Params:
    greedy: bool


BS, LIMIT = 16, 1024
MB = -(-LIMIT // BS)


def expected(chunks, tables_before):
    """Python statement of the layout (the reference's per-token ids, positions and slots,
    runner/model_runner.py:162-205; the plan rows longest first)."""
    b = len(chunks)
    pos = [c.num_computed for c in chunks]
    ids = [c.token_ids[p] for c, p in zip(chunks, pos)]
    slots = [c.block_table[p // BS] * BS + p % BS for c, p in zip(chunks, pos)]
    order = sorted(range(b), key=pos.__getitem__, reverse=True)
    tables = tables_before.copy()
    changed = False
    for r, i in enumerate(order):
        need = (pos[i] + BS) // BS
        row = np.asarray(chunks[i].block_table[:need], dtype=np.int32)
        if not np.array_equal(tables[r * MB : r * MB + need], row):
            tables[r * MB : r * MB + need] = row
            changed = True
    i64 = np.array(ids + pos + slots, dtype=np.int64)
    meta = np.array(order + [pos[i] + 1 for i in order], dtype=np.int32)
    return i64, meta, tables, changed


def buffers(b):
    return np.zeros(3 * b, np.int64), np.zeros(2 * b, np.int32), np.zeros(b * MB, np.int32)


def batch(rng, b, lo=1, hi=LIMIT - 1):
    out = []
    for _ in range(b):
        p = rng.randint(lo, hi)
        table = rng.sample(range(5000), (p + BS) // BS + rng.randint(0, 2))
        out.append(Chunk([rng.randrange(151936) for _ in range(p + 1)], p, 1, table))
    return out


@pytest.mark.parametrize("seed", range(6))
def test_pack_decode_matches_layout(seed):
    rng = random.Random(seed)
    b = rng.choice([1, 5, 64, 129])
    chunks = batch(rng, b, hi=rng.choice([40, LIMIT - 1]))  # short contexts: many tied positions
    hi, hm, ht = buffers(b)
    ei, em, et, ech = expected(chunks, ht)
    rc = _hostprep.pack_decode(chunks, BS, LIMIT, hi, hm, ht, MB)
    assert rc == int(ech) == 1
    np.testing.assert_array_equal(hi, ei)
    np.testing.assert_array_equal(hm, em)
    np.testing.assert_array_equal(ht, et)
    # The next step: every sequence one token further; tables unchanged except where a block starts.
    for c in chunks:
        c.token_ids.append(rng.randrange(151936))
        c.num_computed += 1
        if (c.num_computed + BS) // BS > len(c.block_table):
            c.block_table.append(rng.randrange(5000))
    ei, em, et, ech = expected(chunks, ht)
    rc = _hostprep.pack_decode(chunks, BS, LIMIT, hi, hm, ht, MB)
    assert rc == int(ech)
    np.testing.assert_array_equal(hi, ei)
    np.testing.assert_array_equal(hm, em)
    np.testing.assert_array_equal(ht, et)
    # The same step again: nothing to upload.
    assert _hostprep.pack_decode(chunks, BS, LIMIT, hi, hm, ht, MB) == 0


def test_pack_decode_tuple_sequences_and_greedy_params():
    rng = random.Random(7)
    chunks = batch(rng, 9)
    for c in chunks[:4]:
        c.token_ids, c.block_table, c.params = tuple(c.token_ids), tuple(c.block_table), Params(True)
    hi, hm, ht = buffers(9)
    ei, em, et, _ = expected(chunks, ht)
    assert _hostprep.pack_decode(chunks, BS, LIMIT, hi, hm, ht, MB) == 1
    np.testing.assert_array_equal(hi, ei)
    np.testing.assert_array_equal(hm, em)
    np.testing.assert_array_equal(ht, et)


@pytest.mark.parametrize("case", ["two_new", "not_last", "past_limit", "sampled"])
def test_pack_decode_not_a_decode_step_writes_nothing(case):
    rng = random.Random(3)
    chunks = batch(rng, 6)
    c = chunks[4]
    if case == "two_new":
        c.num_new = 2
    elif case == "not_last":
        c.token_ids.append(1)
    elif case == "past_limit":
        chunks = batch(rng, 6, lo=LIMIT, hi=LIMIT + 5)
    else:
        c.params = Params(False)
    hi, hm, ht = buffers(6)
    hi[:] = 7
    assert _hostprep.pack_decode(chunks, BS, LIMIT, hi, hm, ht, MB) == -1
    assert (hi == 7).all() and not hm.any() and not ht.any()


def test_pack_decode_errors_leave_buffers_alone():
    rng = random.Random(4)
    chunks = batch(rng, 5)
    hi, hm, ht = buffers(5)
    short = chunks[3]
    short.block_table = short.block_table[: short.num_computed // BS]  # one block short
    with pytest.raises(RuntimeError, match="shorter than context"):
        _hostprep.pack_decode(chunks, BS, LIMIT, hi, hm, ht, MB)
    assert not hi.any() and not hm.any() and not ht.any()
    chunks = batch(rng, 5)
    chunks[2].block_table[0] = 2**31
    with pytest.raises(OverflowError):
        _hostprep.pack_decode(chunks, BS, LIMIT, hi, hm, ht, MB)
    assert not hi.any() and not hm.any() and not ht.any()
    with pytest.raises(ValueError, match="too small"):
        _hostprep.pack_decode(chunks, BS, LIMIT, hi[:5], hm, ht, MB)


def test_pack_decode_empty_batch():
    hi, hm, ht = buffers(0)
    assert _hostprep.pack_decode([], BS, LIMIT, hi, hm, ht, MB) == 0


# ---- pack_step: the flat batch and the attention plan of an eager step ----------------------------

import torch  # noqa: E402

from miniserve_amd.attention.backends import PREFILL_TILE_SIZES, SeqChunk, build_attention_metadata  # noqa: E402
from miniserve_amd.runner.model_runner import ModelRunner  # noqa: E402


def flat_batch(chunks):
    """Python statement of the flat batch (runner/model_runner.py:162-205): ids, positions, slots,
    the sampled sequences and their last rows, and the SeqChunk list the plan is built from."""
    ids, pos, slots, rows, sample, seqs = [], [], [], [], [], []
    flat = 0
    for idx, s in enumerate(chunks):
        start, n, table = s.num_computed, s.num_new, s.block_table
        for p in range(start, start + n):
            ids.append(s.token_ids[p])
            pos.append(p)
            slots.append(table[p // BS] * BS + p % BS)
        seqs.append(SeqChunk(flat, n, start, list(table)))
        if start + n == len(s.token_ids):
            sample.append(idx)
            rows.append(flat + n - 1)
        flat += n
    return ids, pos, slots, rows, sample, seqs


def mixed_batch(rng, n_dec, prompts, spare=0):
    out = []
    for _ in range(n_dec):
        p = rng.randint(1, 700)
        toks = [rng.randrange(151936) for _ in range(p + 1)]
        out.append(Chunk(toks, p, 1, rng.sample(range(9000), (p + BS) // BS + rng.randint(0, spare))))
    for cached, n, whole in prompts:
        total = cached + n + (0 if whole else rng.randint(1, 40))
        toks = [rng.randrange(151936) for _ in range(total)]
        out.append(Chunk(toks, cached, n, rng.sample(range(9000), -(-(cached + n) // BS) + rng.randint(0, spare))))
    rng.shuffle(out)
    return out


def runner_cpu():
    r = ModelRunner.__new__(ModelRunner)
    r.block_size, r.device, r.max_model_len = BS, torch.device("cpu"), 4096
    return r


@pytest.mark.parametrize("seed", range(5))
def test_pack_step_matches_flat_batch_and_plan(seed):
    rng = random.Random(100 + seed)
    prompts = [(0, 1984, True)] if seed == 0 else [(rng.randint(0, 300), rng.randint(2, 200), rng.random() < 0.5)
                                                  for _ in range(rng.randint(0, 4))]
    chunks = mixed_batch(rng, rng.choice([0, 3, 64]), prompts, spare=2)
    if not chunks:
        chunks = mixed_batch(rng, 2, [])
    r = runner_cpu()
    inp = r.prepare(chunks)
    ids, pos, slots, rows, sample, seqs = flat_batch(chunks)
    assert inp.input_ids.tolist() == ids and inp.positions.tolist() == pos
    assert inp.attn.slot_mapping.tolist() == slots and inp.logits_rows.tolist() == rows and inp.sample_idx == sample
    want = build_attention_metadata(seqs, torch.tensor(slots, dtype=torch.int64), BS, r.split_context)
    for plan, ref in ((inp.attn.decode, want.decode), (inp.attn.prefill, want.prefill)):
        assert (plan is None) == (ref is None)
    if want.decode is not None:
        for name in ("q_rows", "context_lens", "block_tables"):
            assert torch.equal(getattr(inp.attn.decode, name), getattr(want.decode, name)), name
        assert inp.attn.decode.split_context == want.decode.split_context
    if want.prefill is not None:
        assert torch.equal(inp.attn.prefill.seq_info, want.prefill.seq_info)
        assert torch.equal(inp.attn.prefill.block_tables, want.prefill.block_tables)
        assert sorted(inp.attn.prefill.work) == sorted(want.prefill.work) == list(PREFILL_TILE_SIZES)
        for t in PREFILL_TILE_SIZES:
            assert torch.equal(inp.attn.prefill.work[t], want.prefill.work[t]), t


def test_pack_step_errors():
    rng = random.Random(9)
    chunks = mixed_batch(rng, 3, [(16, 40, True)])
    pre = next(c for c in chunks if c.num_new > 1)
    pre.block_table = pre.block_table[:2]
    with pytest.raises(RuntimeError, match="shorter than context"):
        _hostprep.pack_step(chunks, BS, PREFILL_TILE_SIZES)
    chunks = mixed_batch(rng, 3, [])
    chunks[1].num_new = 5  # past the end of its token list
    with pytest.raises(ValueError, match="schedules tokens"):
        _hostprep.pack_step(chunks, BS, PREFILL_TILE_SIZES)
    chunks = mixed_batch(rng, 3, [])
    chunks[2].block_table[0] = -(2**31) - 1
    with pytest.raises(OverflowError):
        _hostprep.pack_step(chunks, BS, PREFILL_TILE_SIZES)


# ---- which decode rows own the slot they write -----------------------------------------------------


def owns_by_positions(chunks):
    """Every (block, offset) of every row's context against every row's new slot."""
    new = [(c.block_table[c.num_computed // BS], c.num_computed % BS) for c in chunks]
    for r, c in enumerate(chunks):
        for p in range(c.num_computed + 1):
            at = (c.block_table[p // BS], p % BS)
            if any(at == s and not (r == w and p == c.num_computed) for w, s in enumerate(new)):
                return False
    return True


@pytest.mark.parametrize("seed", range(40))
def test_rows_own_slots_matches_every_position(seed):
    """Random batches over few blocks (own, shared as full prefixes, shared where they are written, the
    same block twice in one table), through every entry point that answers."""
    rng = random.Random(500 + seed)
    chunks = batch(rng, rng.choice([1, 2, 7, 40]), hi=rng.choice([20, 200]))
    fresh = iter(range(1, 10_000))  # (block 0 is what an unused table entry holds)
    for c in chunks:
        c.block_table = [next(fresh) for _ in c.block_table]
    for _ in range(rng.choice([0, 1, 3])):
        a, b = rng.choice(chunks), rng.choice(chunks)
        n = rng.randint(0, min(len(a.block_table), len(b.block_table)))
        if rng.random() < 0.5:
            a.block_table[:n] = b.block_table[:n]
        else:
            a.block_table[rng.randrange(len(a.block_table))] = rng.choice(b.block_table)
    want = owns_by_positions(chunks)
    assert _hostprep.pack_step(chunks, BS, PREFILL_TILE_SIZES, 128)[4] is want
    assert _hostprep.pack_step(chunks, BS, PREFILL_TILE_SIZES, len(chunks) - 1 or -1)[4:] in ((), (None,))
    hi, hm, ht = buffers(len(chunks))
    rc = _hostprep.pack_decode(chunks, BS, LIMIT, hi, hm, ht, MB, True)
    assert (rc == 1) is want and (want or not (hi.any() or hm.any() or ht.any()))
    assert runner_cpu().prepare(chunks).attn.decode.own_slots is want
    seqs = [SeqChunk(i, 1, c.num_computed, c.block_table) for i, c in enumerate(chunks)]
    meta = build_attention_metadata(seqs, torch.zeros(len(chunks), dtype=torch.int64), BS)
    assert meta.decode.own_slots is (None if want else False)  # the slots themselves are not known there


def test_rows_own_slots_cases():
    def owns(tables, ctx):
        return _hostprep.rows_own_slots(np.array(tables, np.int32), np.array(ctx, np.int32), BS)

    assert owns([[3, 4], [3, 5]], [20, 32])  # a full prefix block shared
    assert not owns([[3, 4], [3, 4]], [20, 21])  # the same sequence at two lengths
    assert not owns([[3, 4], [3, 4]], [20, 20])
    assert not owns([[3, 4], [4, 9]], [20, 17])  # row 0 writes into row 1's first block
    assert owns([[3, 4], [9, 4]], [16, 32])  # row 0 does not reach its second entry
    assert not owns([[3, 3]], [17])  # its own first block
    assert not owns([[-1, 0]], [5])  # read as block 0, never written
    assert owns([], []) and owns([[0, 0]], [0])
    with pytest.raises(ValueError):
        owns([[3, 4]], [33])
