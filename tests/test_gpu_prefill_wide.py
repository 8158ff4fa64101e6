"""GPU parity of prefill attention on 32-query wavefront tiles (msa_paged_attention_prefill_wide) against
the CPU oracle and the 16-query kernel, and of the rule that picks between them.

Both kernels round the same values (scores in float32, probabilities to bf16, their sums over the
rounded ones), in another order only where key groups merge: within rel-L2 2e-3 of each other and, as
the 16-query kernel, 1e-2 of the oracle. Lengths cover single tokens, the edges of the 32-query tile and
of the 32-key tile, cached tokens off block and tile boundaries, and every group size."""

from __future__ import annotations

import pytest
import torch
from helpers import rel_l2

from miniserve_amd import kernels
from miniserve_amd.attention import backends as ab
from oracle import attention as oa

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")


def _case(heads, kv_heads, seqs, seed):
    g = torch.Generator().manual_seed(seed)
    need = [-(-(c + n) // 16) for c, n in seqs]
    perm = torch.randperm(sum(need) + 3, generator=g).tolist()
    chunks, flat, off = [], 0, 0
    for (c, n), b in zip(seqs, need):
        chunks.append((flat, n, c, perm[off : off + b]))
        flat, off = flat + n, off + b

    def t(*shape):
        return torch.randn(*shape, generator=g).to(torch.bfloat16)

    return (chunks, t(flat, heads, 128), t(flat, kv_heads, 128), t(flat, kv_heads, 128),
            t((sum(need) + 3) * 16, kv_heads, 128), t((sum(need) + 3) * 16, kv_heads, 128))


def _slots(chunks):
    return torch.tensor([tab[p // 16] * 16 + p % 16 for _, n, c, tab in chunks for p in range(c, c + n)])


@pytest.mark.parametrize("heads,kv_heads,seqs", [
    (4, 1, [(0, 31), (0, 32), (0, 33)]),
    (4, 1, [(0, 2), (17, 5), (95, 64), (96, 65)]),
    (8, 4, [(0, 63), (0, 64), (1, 65), (300, 2)]),
    (8, 4, [(31, 129), (700, 40)]),
    (3, 3, [(0, 127), (0, 128), (5, 129)]),
    (16, 4, [(500, 200)]),
])
def test_prefill_wide_matches(heads, kv_heads, seqs):
    chunks, q, k, v, kc, vc = _case(heads, kv_heads, seqs, seed=heads + len(seqs))
    slots = _slots(chunks)
    kc[slots], vc[slots] = k, v
    meta = ab.build_attention_metadata([ab.SeqChunk(*c) for c in chunks], slots.to(DEV), 16)
    p, tile = meta.prefill, ab.PREFILL_TILE[heads // kv_heads]
    qd, kd, vd = q.to(DEV), kc.to(DEV), vc.to(DEV)
    outs = []
    for wide in (False, True):
        out = torch.zeros_like(qd)
        kernels.paged_attention_prefill(qd, kd, vd, p.block_tables, p.seq_info, p.work[2 * tile if wide else tile],
                                        128**-0.5, out, 16, wide)
        outs.append(out.cpu())
    assert rel_l2(outs[1], outs[0]) < 2e-3
    om = oa.build_attention_metadata([oa.SeqChunk(*c) for c in chunks], slots, 16)
    ref = oa.paged_attention(q, k, v, kc.clone(), vc.clone(), om, 128**-0.5)
    assert rel_l2(outs[1], ref) < 1e-2


@pytest.mark.parametrize("heads,kv_heads,seqs,wide", [
    (32, 8, [(0, 1536)], True),  # 48 tiles of 32 x 8 heads
    (32, 8, [(0, 1504)], False),
    (8, 8, [(0, 128)] * 48, True),
    (32, 8, [(100, 4)] * 64, False),  # half-empty tiles
])
def test_prefill_wide_rule(heads, kv_heads, seqs, wide):
    chunks, q, k, v, kc, vc = _case(heads, kv_heads, seqs, seed=7)
    slots = _slots(chunks).to(DEV)
    meta = ab.build_attention_metadata([ab.SeqChunk(*c) for c in chunks], slots, 16)
    p, tile = meta.prefill, ab.PREFILL_TILE[heads // kv_heads]
    assert ab.prefill_takes_wide(p, tile, kv_heads) is wide
    qd, kd, vd = q.to(DEV), kc.to(DEV), vc.to(DEV)
    out = ab.paged_attention(qd, k.to(DEV), v.to(DEV), kd, vd, meta, 128**-0.5)
    ref = torch.zeros_like(qd)
    kernels.paged_attention_prefill(qd, kd, vd, p.block_tables, p.seq_info, p.work[tile], 128**-0.5, ref, 16)
    assert rel_l2(out.cpu(), ref.cpu()) < 2e-3


@pytest.mark.parametrize("heads,kv_heads", [(8, 8), (16, 8), (32, 8)])
def test_prefill_wide_past_4gb_of_cache(heads, kv_heads):
    """A cache of 4 GB and more is addressed with 64-bit offsets: blocks at the end of such a pool give, bit
    for bit, what the same blocks give in a small one. The rest of the large pool is not read."""
    chunks, q, k, v, kc, vc = _case(heads, kv_heads, [(70, 150), (0, 40), (33, 129)], seed=heads)
    slots = _slots(chunks)
    kc[slots], vc[slots] = k, v
    base = (1 << 32) // (16 * kv_heads * 128 * 2) + 4096 - kc.shape[0] // 16
    tile, qd, outs = ab.PREFILL_TILE[heads // kv_heads], q.to(DEV), []
    for at in (0, base):
        big = [torch.empty(at * 16 + kc.shape[0], kv_heads, 128, dtype=torch.bfloat16, device=DEV) for _ in range(2)]
        big[0][at * 16 :], big[1][at * 16 :] = kc.to(DEV), vc.to(DEV)
        assert (big[0].numel() * 2 > 1 << 32) is (at > 0)
        meta = ab.build_attention_metadata([ab.SeqChunk(f, n, c, [b + at for b in t]) for f, n, c, t in chunks],
                                           (slots + at * 16).to(DEV), 16)
        p, out = meta.prefill, torch.zeros_like(qd)
        kernels.paged_attention_prefill(qd, *big, p.block_tables, p.seq_info, p.work[2 * tile], 128**-0.5, out, 16, True)
        outs.append(out.cpu())
        del big
    assert torch.equal(*outs) and outs[0].abs().sum() > 0
    torch.cuda.empty_cache()
