"""GPU parity of the sampling kernel (top-k / top-p without a sort, temperature, the exponential
race) against the sampling oracle and a float64 brute force on the same logits and noise.

Bars: kept masks identical to the float64 brute force (and the oracle) on every row whose top-p
cut is decidable (no cumulative probability within 1e-5 of 1 - p); on the other rows (a cut in the
dense tail of a 151,936-entry vocabulary, where the reference's own float32 cumsum decides by
rounding) only tokens within 1e-5 of the cut may differ; probabilities within rel-L2 1e-5 of the
oracle's on decidable rows; sampled ids equal to the oracle's given the same noise wherever the
best two scores differ by more than 1e-4 relative; the reference's own unit cases exactly.
"""

from __future__ import annotations

from dataclasses import dataclass

import numpy as np
import pytest
import torch
from helpers import rel_l2
from test_oracle_sampler import CHI2_DF4_P001, brute_force_cut, brute_force_mask, chi_square

from miniserve_amd import kernels
from miniserve_amd.runner import sampler as hs
from oracle import sampler as osm

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")


@dataclass
class Params:
    temperature: float = 1.0
    top_p: float = 1.0
    top_k: int = -1

    @property
    def greedy(self) -> bool:
        return self.temperature < 1e-5


def _case(rows, vocab, seed):
    g = torch.Generator().manual_seed(seed)
    logits = torch.randn(rows, vocab, generator=g) * 3
    k = torch.randint(1, 200, (rows,), generator=g).to(torch.int32)
    k[::4] = vocab  # every fourth row: no top-k
    p = (torch.rand(rows, generator=g) * 0.9 + 0.05).float()
    p[1::4] = 1.0  # no top-p
    return logits, k, p


def test_reference_unit_cases():
    logits = torch.tensor([[1.0, 4.0, 3.0, 2.0, 0.0]], device=DEV)
    kept = hs.apply_top_k_top_p(logits, torch.tensor([2]), torch.tensor([1.0])) > float("-inf")
    assert kept.cpu().tolist() == [[False, True, True, False, False]]
    kept = hs.apply_top_k_top_p(logits, torch.tensor([5]), torch.tensor([0.8])) > float("-inf")
    assert kept.cpu().tolist() == [[False, True, True, False, False]]
    x = torch.randn(6, 50, generator=torch.Generator().manual_seed(1)).to(DEV)
    assert torch.equal(hs.sample(x, [Params(temperature=0)] * 6, [None] * 6), x.argmax(-1))
    y = torch.randn(4, 100, generator=torch.Generator().manual_seed(2)).to(DEV)
    params = [Params(top_k=1), Params(top_p=1e-6)] * 2
    assert torch.equal(hs.sample(y, params, [None] * 4), y.argmax(-1))


@pytest.mark.parametrize("rows,vocab", [(64, 151936), (33, 5000), (8, 64)])
def test_masks_match_float64_brute_force(rows, vocab):
    logits, k, p = _case(rows, vocab, seed=vocab)
    got = kernels.top_k_top_p_mask(logits.to(DEV), k.to(DEV), p.to(DEV)).cpu()
    ref = osm.apply_top_k_top_p(logits, k.long(), p)
    exact = 0
    for r in range(rows):
        kept = got[r] > float("-inf")
        assert torch.equal(got[r][kept], logits[r][kept])  # kept values untouched
        mask, boundary = brute_force_cut(logits[r].double().numpy(), int(k[r]), float(p[r]), tol=1e-5)
        if not boundary.any():  # decidable: identical to the brute force and to the oracle
            assert np.array_equal(kept.numpy(), mask), r
            assert torch.equal(kept, ref[r] > float("-inf")), r
            exact += 1
        else:  # a cut inside the dense tail: only tokens at the cut may fall either way
            differ = kept.numpy() != mask
            assert not (differ & ~boundary).any(), (r, int(differ.sum()))
    assert exact >= rows // 2


def test_probs_match_the_oracle():
    rows, vocab = 48, 151936
    logits, k, p = _case(rows, vocab, seed=3)
    temps = (torch.rand(rows, generator=torch.Generator().manual_seed(4)) * 1.5 + 0.2).float()
    got = kernels.sampling_probs(logits.to(DEV), temps.to(DEV), k.to(DEV), p.to(DEV)).cpu()
    ref = osm.compute_probs(logits, temps, k.long(), p)
    for r in range(rows):
        z = (logits[r] / temps[r]).double().numpy()
        _, ok = brute_force_mask(z, int(k[r]), float(p[r]))
        if ok:
            assert rel_l2(got[r], ref[r]) < 1e-5, r
    assert torch.allclose(got.sum(-1), torch.ones(rows), atol=1e-5)


def test_sampled_ids_match_the_oracle_with_the_same_noise():
    rows, vocab = 64, 151936
    logits, k, p = _case(rows, vocab, seed=5)
    temps = torch.full((rows,), 0.8)
    greedy = torch.zeros(rows, dtype=torch.bool)
    greedy[::8] = True
    noise = torch.empty(rows, vocab).exponential_(generator=torch.Generator().manual_seed(6))
    got = kernels.sample_ids(logits.to(DEV), temps.to(DEV), k.to(DEV), p.to(DEV), greedy.to(torch.uint8).to(DEV),
                             noise.to(DEV)).cpu()
    ref = osm.sample(logits, temps, k.long(), p, greedy, noise)
    probs = osm.compute_probs(logits, temps, k.long(), p)
    checked = 0
    for r in range(rows):
        z = (logits[r] / temps[r]).double().numpy()
        _, ok = brute_force_mask(z, int(k[r]), float(p[r]))
        s = (probs[r] / noise[r]).double()
        top2 = s.topk(2).values
        if greedy[r] or (ok and float(top2[0] - top2[1]) > 1e-4 * float(top2[0])):
            assert int(got[r]) == int(ref[r]), r
            checked += 1
    assert checked >= rows * 3 // 4


def test_sampling_distribution_and_seeded_rows():
    rows = 100_000
    logits = torch.tensor([[0.5, 1.5, -1.0, 0.0, 1.0]], device=DEV).repeat(rows, 1)
    torch.manual_seed(0)
    tokens = hs.sample(logits, [Params(temperature=1.0)] * rows, [None] * rows)
    counts = torch.bincount(tokens.cpu(), minlength=5).double()
    assert chi_square(counts, logits[0].cpu().double().softmax(-1)) < CHI2_DF4_P001
    x = torch.randn(3, 1000, generator=torch.Generator().manual_seed(7)).to(DEV)
    params = [Params(temperature=1.0)] * 3

    def gens():
        return [torch.Generator(device=DEV).manual_seed(7) for _ in range(3)]

    assert torch.equal(hs.sample(x, params, gens()), hs.sample(x, params, gens()))


def test_edge_rows():
    """-inf entries, every value equal with top-k (the ties at the k-th value are all kept, as
    `sorted < kth` keeps them), k = vocab - 1, p just below 1."""
    vocab = 1000
    x = torch.randn(4, vocab, generator=torch.Generator().manual_seed(8))
    x[0, ::3] = float("-inf")
    x[1] = 0.25
    k = torch.tensor([10, 3, vocab - 1, vocab], dtype=torch.int32)
    p = torch.tensor([1.0, 1.0, 1.0, 0.999])
    got = kernels.top_k_top_p_mask(x.to(DEV), k.to(DEV), p.to(DEV)).cpu()
    ref = osm.apply_top_k_top_p(x, k.long(), p)
    assert torch.equal(got[0] > float("-inf"), ref[0] > float("-inf"))
    assert bool((got[1] > float("-inf")).all()) and bool((ref[1] > float("-inf")).all())
    assert torch.equal(got[2] > float("-inf"), ref[2] > float("-inf"))
    mask, ok = brute_force_mask(x[3].double().numpy(), vocab, 0.999)
    assert not ok or np.array_equal((got[3] > float("-inf")).numpy(), mask)


def _whole_row_ids(logits, temps, k, p, greedy, noise):
    """msa_sample without a workspace: one workgroup per row over the whole vocabulary."""
    from miniserve_amd import _native

    r, v = logits.shape
    out = torch.empty(r, dtype=torch.int64, device=DEV)
    _native.call("msa_sample", logits.data_ptr(), logits.stride(0), r, v, temps.data_ptr(), k.data_ptr(),
                 p.data_ptr(), greedy.data_ptr(), noise.data_ptr(), noise.stride(0), out.data_ptr(), None, 0,
                 torch.cuda.current_stream().cuda_stream)
    return out


@pytest.mark.parametrize("vocab", [151936, 10240, 10241, 70000, 200000, 400000])
def test_chunked_sampling_matches_the_whole_row_path(vocab):
    """The chunked path (greedy rows and 0 < top_k <= 256 over vocabulary chunks) against the
    whole-row path on the same logits and noise: identical ids wherever the best two scores differ
    by more than 1e-5 relative (they sum Z in different orders). Rows: greedy, top-k 1..256 with
    and without top-p, top-k above 256 and none (whole-row fallback inside the call), and rows of
    rounded logits whose ties at the k-th value overflow a chunk's candidates (fallback) or fill
    the finishing workgroup's bound (the radix path). Vocabularies: one chunk, a ragged last chunk,
    up to 16 chunks and up to 32 (candidates gathered in registers), 40 (gathered through LDS)."""
    rows = 48
    g = torch.Generator().manual_seed(vocab)
    logits = torch.randn(rows, vocab, generator=g) * 3
    logits[40:] = torch.round(logits[40:])  # many equal values: ties at the cut
    k = torch.randint(1, 257, (rows,), generator=g).to(torch.int32)
    k[5] = 1
    k[6] = 256
    k[7] = 300  # above the chunked range
    k[8] = vocab  # no top-k
    p = (torch.rand(rows, generator=g) * 0.9 + 0.05).float()
    p[::3] = 1.0
    temps = (torch.rand(rows, generator=g) * 1.2 + 0.3).float()
    greedy = torch.zeros(rows, dtype=torch.uint8)
    greedy[::11] = 1
    noise = torch.empty(rows, vocab).exponential_(generator=g)
    ld, td, kd, pd, gd, nd = (t.to(DEV) for t in (logits, temps, k, p, greedy, noise))
    got = kernels.sample_ids(ld, td, kd, pd, gd, nd).cpu()
    whole = _whole_row_ids(ld, td, kd, pd, gd, nd).cpu()
    again = kernels.sample_ids(ld, td, kd, pd, gd, nd).cpu()
    assert torch.equal(got, again)  # deterministic
    probs = osm.compute_probs(logits, temps, k.long(), p)
    checked = 0
    for r in range(rows):
        if greedy[r]:
            assert int(got[r]) == int(logits[r].argmax()), r
            checked += 1
            continue
        s = (probs[r] / noise[r].clamp_min(1.17549435e-38)).double()
        top2 = s.topk(2).values
        if float(top2[0] - top2[1]) > 1e-5 * float(top2[0]):
            assert int(got[r]) == int(whole[r]), r
            checked += 1
    assert checked >= rows * 3 // 4


@pytest.mark.parametrize("vocab", [64, 10240, 10241, 151936, 660000])
def test_rows_without_top_k_over_chunks(vocab):
    """Rows with temperature alone or top-p alone (mass histogram, cut bin, race over chunks)
    against the whole-row path on the same logits and noise: identical ids wherever the best two
    scores differ by more than 1e-5 relative (float32 scores, each within a few 2^-24 of exact).
    Rows: dense and bf16-rounded logits (ties at the cut), a flat row and a row of few values (more
    entries at the cut than the lists hold), a row with one dominating entry, rows with -inf
    entries, with whole chunks of them and with a NaN, top-p near 0 and near 1, a temperature so
    small that z leaves the range of whole numbers, a row stride that is not the vocabulary.
    Vocabularies: less than a workgroup, one chunk, a one-entry last chunk, 15 chunks, and more
    chunks than the finishing workgroup gathers."""
    rows = 24
    g = torch.Generator().manual_seed(vocab + 1)
    logits = (torch.randn(rows, vocab + 3, generator=g) * 3)[:, :vocab]
    logits[8:14] = logits[8:14].to(torch.bfloat16).float()
    logits[14] = 0.5
    logits[15] = torch.round(logits[15] / 4)
    logits[16, vocab // 2] = 60.0
    logits[17, ::2] = float("-inf")
    logits[18, : vocab - 5] = float("-inf")
    logits[19, 7] = float("nan")
    p = (torch.rand(rows, generator=g) * 0.9 + 0.05).float()
    p[::3] = 1.0
    p[1], p[8], p[17], p[18] = 1e-7, 0.99999, 0.9, 0.7
    temps = (torch.rand(rows, generator=g) * 1.2 + 0.3).float()
    temps[20], temps[22] = 1e-5, 1e-5
    k = torch.full((rows,), vocab, dtype=torch.int32)
    k[2::5] = -1
    greedy = torch.zeros(rows, dtype=torch.uint8)
    greedy[5] = 1
    noise = torch.empty(rows, vocab).exponential_(generator=g)
    ld = torch.empty(rows, vocab + 3, device=DEV)[:, :vocab].copy_(logits)
    td, kd, pd, gd, nd = (t.to(DEV) for t in (temps, k, p, greedy, noise))
    got = kernels.sample_ids(ld, td, kd, pd, gd, nd, wide=True).cpu()
    assert torch.equal(got, kernels.sample_ids(ld, td, kd, pd, gd, nd, wide=True).cpu())  # deterministic
    assert torch.equal(got[greedy.bool()], logits.argmax(-1)[greedy.bool()])
    whole = _whole_row_ids(ld, td, kd, pd, gd, nd).cpu()
    scores = (kernels.sampling_probs(ld, td, kd, pd) / nd.clamp_min(1.17549435e-38)).double()
    top2 = scores.topk(2).values.cpu()
    checked = 0
    for r in range(rows):
        if r == 19 or float(top2[r, 0] - top2[r, 1]) > 1e-5 * float(top2[r, 0]):
            assert int(got[r]) == int(whole[r]), r
            checked += 1
    assert checked >= rows - 2
    none = kernels.sample_ids(ld, td, None, None, gd, nd, wide=True).cpu()  # no filters at all: temperature alone
    full = kernels.sample_ids(ld, td, kd, torch.ones_like(pd), gd, nd, wide=True).cpu()
    assert torch.equal(none, full)


@pytest.mark.parametrize("vocab", [10240, 70000, 151936])
def test_top_p_cut_of_rows_without_top_k(vocab):
    """Where top-p alone cuts, to the resolution the masses are held in: values whose mass at or below
    them, known in float64, lies just above 1 - p (kept) or just below it (dropped), each shown by a noise
    that lets one of its entries win if it is kept. Logits are multiples of 2^-10, so every z - m is exact
    in float32; what is left, relative to the row's total, is B = (entries at or below + 512 bins) masses
    truncated to 2^-44 of the largest entry and 2^-22 of the mass itself (exp within an ulp on both
    sides). Probes lie between B and 3 B off, the kept ones where masses in steps of 2^-40, which lose
    2^-41 an entry on average, would drop them."""
    g = torch.Generator(device=DEV).manual_seed(vocab)
    probes, expect = [], []
    for top in (12.0, 13.0, 14.0):
        z = torch.round(torch.randn(vocab, generator=g, device=DEV) * 1024) / 1024
        z[vocab // 3] = top
        values, group, count = z.unique(return_inverse=True, return_counts=True)
        mass = torch.exp(values.double() - top) * count
        share, below = mass.cumsum(0) / mass.sum(), count.cumsum(0)
        bound = (below + 512) * 2.0**-44 / mass.sum() + 2.0**-22 * share
        for step in (-1, 0, 1):  # the float32 p nearest to 1 - share and its neighbours
            p = (1 - share).float() + step * 2.0**-24
            off = share - (1 - p.double())
            usable = (share > 1e-5) & (share < 0.02) & (off.abs() > bound) & (off.abs() < 3 * bound)
            usable &= (off < 0) | (off < 0.7 * below * 2.0**-41 / mass.sum())
            for j in usable.nonzero().flatten().tolist()[::3][:30]:
                probes.append((z, int((group == j).nonzero()[0]), float(p[j])))
                expect.append(bool(off[j] > 0))
    assert sum(expect) >= 3 and len(expect) - sum(expect) >= 3
    want = torch.tensor(expect)
    logits = torch.stack([z for z, _, _ in probes])
    at = torch.tensor([i for _, i, _ in probes], device=DEV)
    p = torch.tensor([q for _, _, q in probes], device=DEV)
    noise = torch.ones_like(logits).scatter_(1, at[:, None], 1e-30)
    greedy = torch.zeros(len(probes), dtype=torch.uint8, device=DEV)
    got = kernels.sample_ids(logits, torch.ones_like(p), None, p, greedy, noise) == at
    assert torch.equal(got.cpu(), want), (got.cpu() != want).nonzero().flatten().tolist()


def test_calls_spread_only_rows_without_top_k(monkeypatch):
    """The two launches that spread rows without top-k are made where some row gains by them: not for calls
    with a top_k tensor that do not ask for them, nor for batches whose rows are greedy, have top-k
    (of any size), or are short and without top-p; one workgroup a row gives the same ids."""
    from miniserve_amd import _native

    calls, real = [], _native.call

    def record(name, *args):
        calls.append(name)
        real(name, *args)

    monkeypatch.setattr(_native, "call", record)
    small, large = kernels.SAMPLE_WIDE_MIN_VOCAB - 1, kernels.SAMPLE_WIDE_MIN_VOCAB
    for params, vocab, want in [
        ([Params(top_k=20, top_p=0.9), Params(temperature=0.0)], large, "msa_sample"),
        ([Params(top_k=1000), Params(top_k=5)], large, "msa_sample"),
        ([Params()], small, "msa_sample"),
        ([Params(), Params(top_k=20, top_p=0.9)], small, "msa_sample"),
        ([Params(top_k=5), Params()], large, "msa_sample_wide"),
        ([Params(top_p=0.9), Params(top_k=5)], small, "msa_sample_wide"),
        ([Params(temperature=0.0)] * 2, large, "msa_sample"),
    ]:
        x = torch.randn(len(params), vocab, generator=torch.Generator().manual_seed(vocab)).to(DEV)
        torch.cuda.manual_seed(3)
        ids = hs.sample(x, params, [None] * len(params))
        assert calls.pop() == want, (params, vocab)
        if all(p.greedy for p in params):
            continue
        torch.cuda.manual_seed(3)
        noise = torch.empty_like(x).exponential_()
        temps = torch.tensor([max(p.temperature, 1e-5) for p in params], device=DEV)
        k = torch.tensor([p.top_k for p in params], dtype=torch.int32, device=DEV)
        p = torch.tensor([p.top_p for p in params], device=DEV)
        greedy = torch.tensor([p.greedy for p in params], dtype=torch.uint8, device=DEV)
        assert torch.equal(ids, kernels.sample_ids(x, temps, k, p, greedy, noise)) and calls.pop() == "msa_sample"
    noise = torch.empty_like(x).exponential_()
    kernels.sample_ids(x[:, :small], temps, None, p, greedy, noise[:, :small])
    kernels.sample_ids(x[:, :small], temps, None, None, greedy, noise[:, :small])
    assert calls[-2:] == ["msa_sample_wide", "msa_sample"]
