"""GPU parity of the LDS-tiled int8 MFMA GEMM (prefill-sized batches, msa_int8_gemm and the
msa_int8_linear route for 128+ rows) against the CPU oracle on the same seeded inputs.

Bars: within rel-L2 1e-2 of the oracle's bf16 path and within bf16 rounding (4e-3) of a float64
product of the same dequantized weights; deterministic; residual and silu * up epilogues."""

from __future__ import annotations

import pytest
import torch
from helpers import rel_l2

from miniserve_amd import _native, kernels
from oracle import int8 as oi
from oracle import layers as ol

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")


def _bf16(shape, seed, std=1.0):
    return (torch.randn(shape, generator=torch.Generator().manual_seed(seed)) * std).to(torch.bfloat16)


# Split-K (float32 partials merged in split order) serves the shapes with fewer than 192 output
# tiles of 128 x 128 and more than one 512-wide split of K: every shape below but the one-step
# ragged-N one. From 192 tokens up, where 2-16 splits of 1024+ keys fill the chip, the partials
# come from 256 x 128 tiles (eight wavefronts per workgroup), else from 128 x 128 tiles in 2-8
# splits.
GEMM_SHAPES = [
    (256, 6144, 4096),  # Qwen3-8B qkv at 256 decode tokens (split 4)
    (256, 4096, 12288),  # Qwen3-8B down_proj at 256 decode tokens
    (128, 4096, 1024),  # qkv at the GEMM threshold
    (2048, 1024, 2048),  # o_proj of the 2048-token chunked-prefill step
    (300, 1024, 3072),  # ragged M (not a multiple of the 128-token tile)
    (256, 4096, 4096),  # Qwen3-8B o_proj at 256 decode tokens
    (129, 200, 64),  # ragged N (not a multiple of the 128-row tile), one K step
    (1000, 512, 12288),  # K of the Qwen3-8B down_proj
]


@pytest.mark.parametrize("m,n,k", GEMM_SHAPES)
def test_gemm_parity(m, n, k):
    q, s = oi.quantize_int8(_bf16((n, k), seed=n + k, std=0.02))
    x = _bf16((m, k), seed=m)
    xd, qd, sd = x.to(DEV), q.to(DEV), s.to(DEV)  # kept alive: the C call takes raw pointers
    y = kernels.int8_linear(xd, qd, sd)  # the GEMM route (m >= 128), split-K when the tiles are few
    assert torch.equal(y, kernels.int8_linear(xd, qd, sd))  # deterministic
    y2 = torch.empty_like(y)
    _native.call("msa_int8_gemm", kernels._ptr(xd), m, k, k, kernels._ptr(qd), kernels._ptr(sd), n, kernels._ptr(y2),
                 n, 0, None, 0, kernels._stream(y2))  # no workspace: never split
    if _native.query("msa_int8_linear_workspace_size", m, n, k) == 0:
        assert torch.equal(y, y2)
    else:  # split-K sums the same products in another order: bf16 outputs within a rounding step
        assert rel_l2(y.cpu(), y2.cpu()) < 2e-3
    ref = oi.int8_linear(x, q, s)
    exact = x.double() @ oi.dequantize(q, s, torch.bfloat16).double().T
    assert rel_l2(y.cpu(), ref) < 1e-2
    assert rel_l2(y.cpu(), exact) < 4e-3


# Unsplit GEMMs with 128+ output tiles of 256 x 256 that keep at least as many of the 256 CUs'
# workgroup slots busy as the 128 x 128 tiling take the 256 x 256-tile kernel: full, ragged-M,
# ragged-N, one- and three-step K, strided x, all three epilogues.
GEMM256_SHAPES = [
    (2048, 5120, 1024),  # 160 tiles
    (1900, 5000, 192),  # ragged M and N, three K steps
    (2100, 5000, 64),  # one K step, a ninth token block of 52 rows
    (4096, 4096, 1024),  # 256 tiles: 32 per XCD
]


@pytest.mark.parametrize("m,n,k", GEMM256_SHAPES)
@pytest.mark.parametrize("ldx_pad", [0, 64])
def test_gemm256_parity(m, n, k, ldx_pad):
    q, s = oi.quantize_int8(_bf16((n, k), seed=n + k + 1, std=0.02))
    x = _bf16((m, k + ldx_pad), seed=m + 9)
    xd, qd, sd = x.to(DEV), q.to(DEV), s.to(DEV)
    assert _native.query("msa_int8_linear_workspace_size", m, n, k) == 0  # never split
    y = torch.empty((m, n), dtype=torch.bfloat16, device=DEV)
    args = (kernels._ptr(xd), m, k, k + ldx_pad, kernels._ptr(qd), kernels._ptr(sd), n)
    _native.call("msa_int8_gemm", *args, kernels._ptr(y), n, 0, None, 0, kernels._stream(y))
    y2 = torch.empty_like(y)
    _native.call("msa_int8_gemm", *args, kernels._ptr(y2), n, 0, None, 0, kernels._stream(y2))
    assert torch.equal(y, y2)  # deterministic
    xv = x[:, :k]
    ref = oi.int8_linear(xv, q, s)
    exact = xv.double() @ oi.dequantize(q, s, torch.bfloat16).double().T
    assert rel_l2(y.cpu(), ref) < 1e-2
    assert rel_l2(y.cpu(), exact) < 4e-3
    if ldx_pad == 0:  # the model's route: same kernel
        assert torch.equal(y, kernels.int8_linear(xd, qd, sd))
    # residual epilogue in place: exact add on the kernel's own product
    r = _bf16((m, n), seed=m + 10)
    rd = r.to(DEV)
    _native.call("msa_int8_gemm", *args, kernels._ptr(rd), n, 2, kernels._ptr(rd), n, kernels._stream(rd))
    assert torch.equal(rd.cpu(), r + y.cpu())


@pytest.mark.parametrize("m,half,k", [
    (2048, 3072, 1024), (2000, 2600, 128), (2304, 2560, 64),
    (250, 8200, 2112),  # 129 tiles of 128 rows, a longer K: sixteen wavefronts
    (1000, 3072, 1024), (1300, 8190, 64),  # eight: 192 tiles, 768
])
def test_gemm256_silu_mul(m, half, k):
    n = 2 * half
    q, s = oi.quantize_int8(_bf16((n, k), seed=m + half, std=0.02))
    x = _bf16((m, k), seed=m + 4)
    y = kernels.int8_linear(x.to(DEV), q.to(DEV), s.to(DEV), epilogue=kernels.EPI_SILU_MUL)
    assert y.shape == (m, half)
    gate, up = oi.int8_linear(x, q, s).chunk(2, dim=-1)
    assert rel_l2(y.cpu(), torch.nn.functional.silu(gate) * up) < 1e-2
    g64, u64 = (x.double() @ oi.dequantize(q, s, torch.bfloat16).double().T).chunk(2, dim=-1)
    assert rel_l2(y.cpu(), torch.nn.functional.silu(g64) * u64) < 8e-3


@pytest.mark.parametrize("m", [128, 333, 2048])
def test_gemm_silu_mul(m):
    n, k = 6144, 1024
    q, s = oi.quantize_int8(_bf16((n, k), seed=m, std=0.02))
    x = _bf16((m, k), seed=m + 1)
    y = kernels.int8_linear(x.to(DEV), q.to(DEV), s.to(DEV), epilogue=kernels.EPI_SILU_MUL)
    gate, up = oi.int8_linear(x, q, s).chunk(2, dim=-1)
    ref = torch.nn.functional.silu(gate) * up
    assert y.shape == (m, n // 2)
    assert rel_l2(y.cpu(), ref) < 1e-2


@pytest.mark.parametrize("m,k", [(128, 3072), (2048, 2048)])
def test_gemm_residual_in_place(m, k):
    n = 1024
    q, s = oi.quantize_int8(_bf16((n, k), seed=k, std=0.02))
    x = _bf16((m, k), seed=m + 2)
    r = _bf16((m, n), seed=m + 3)
    rd = r.to(DEV)
    kernels.int8_linear(x.to(DEV), q.to(DEV), s.to(DEV), epilogue=kernels.EPI_RESIDUAL, residual=rd, out=rd)
    y = kernels.int8_linear(x.to(DEV), q.to(DEV), s.to(DEV)).cpu()
    assert torch.equal(rd.cpu(), r + y)  # the add itself is exact on the kernel's own product
    assert rel_l2(rd.cpu(), r + oi.int8_linear(x, q, s)) < 1e-2


@pytest.mark.parametrize("m,n,k", [(2048, 1024, 2048), (2048, 1024, 3072), (256, 4096, 4096), (128, 1024, 3072),
                                   (300, 2048, 1024), (64, 1024, 1024)])
def test_linear_add_rmsnorm(m, n, k):
    """o / down projection + residual + the next RMSNorm in one call (split-K partials merged, added
    and normalized by one kernel when the GEMM splits) against the unfused linear and norm."""
    q, s = oi.quantize_int8(_bf16((n, k), seed=n + 2 * k, std=0.02))
    x = _bf16((m, k), seed=m + 5)
    r = _bf16((m, n), seed=m + 6)
    w = (1 + 0.1 * torch.randn(n, generator=torch.Generator().manual_seed(7))).to(torch.bfloat16)
    xd, qd, sd, wd = x.to(DEV), q.to(DEV), s.to(DEV), w.to(DEV)
    r1 = r.to(DEV)
    h1 = kernels.int8_linear_add_rmsnorm(xd, qd, sd, r1, wd, 1e-6)
    r2 = r.to(DEV)
    kernels.int8_linear(xd, qd, sd, kernels.EPI_RESIDUAL, residual=r2, out=r2)
    h2 = kernels.rmsnorm(r2, wd, 1e-6)
    assert torch.equal(r1, r2)  # the merge sums the partials in the same split order
    assert rel_l2(h1.cpu(), h2.cpu()) < 2e-3  # sums of squares in another float32 order
    ref = ol.rms_norm(r + oi.int8_linear(x, q, s), w, 1e-6)
    assert rel_l2(h1.cpu(), ref) < 1e-2


@pytest.mark.parametrize("m,heads,kv_heads,k", [(2048, 16, 8, 1024), (300, 32, 8, 1024), (129, 8, 8, 2048)])
def test_gemm_qk_norm_rope_cache_matches_unfused(m, heads, kv_heads, k):
    """The qkv GEMM with the q/k-norm + RoPE + cache write fused after it (in its epilogue at 2048
    tokens; split-K partials summed by the q/k-norm kernel at 300 and 129, where the GEMM splits)
    against the plain linear on the same route followed by the standalone kernel (pinned against
    the oracle in test_gpu_kernels.py): the same q and caches bit for bit, including skipped slots
    (-1 and past the pool); and q within the oracle's bar."""
    d = 128
    n = (heads + 2 * kv_heads) * d
    qw8, sc = oi.quantize_int8(_bf16((n, k), seed=m + heads, std=0.02))
    x = _bf16((m, k), seed=m + 7)
    gen = torch.Generator().manual_seed(m)
    nq = (1 + 0.1 * torch.randn(d, generator=gen)).to(torch.bfloat16)
    nk = (1 + 0.1 * torch.randn(d, generator=gen)).to(torch.bfloat16)
    cos_t, sin_t = ol.rope_tables(d, 4096, 1e6)
    pos = torch.randint(0, 4096, (m,), generator=gen)
    num_slots = m + 64
    slots = torch.randperm(num_slots, generator=gen)[:m]
    slots[3] = -1
    slots[m // 2] = num_slots + 5  # past the pool: skipped
    xd, qd, sd = x.to(DEV), qw8.to(DEV), sc.to(DEV)
    args = (nq.to(DEV), nk.to(DEV), 1e-6, cos_t[pos].contiguous().to(DEV), sin_t[pos].contiguous().to(DEV), slots.to(DEV))
    kc1 = torch.zeros(num_slots, kv_heads, d, dtype=torch.bfloat16, device=DEV)
    vc1, kc2, vc2 = torch.zeros_like(kc1), torch.zeros_like(kc1), torch.zeros_like(kc1)
    splits = _native.query("msa_int8_linear_workspace_size", m, n, k) > 0
    assert splits == (m < 2048)
    q1 = kernels.int8_linear_qk_norm_rope_cache(xd, qd, sd, heads, kv_heads, d, *args, kc1, vc1)
    qkv = kernels.int8_linear(xd, qd, sd)  # the same GEMM route (the same tiles, split or not)
    q2 = kernels.qk_norm_rope_cache(qkv, heads, kv_heads, d, *args, kc2, vc2)
    assert torch.equal(q1, q2)
    assert torch.equal(kc1, kc2) and torch.equal(vc1, vc2)
    assert int(torch.count_nonzero(kc1.abs().sum((1, 2)))) == m - 2  # two rows skipped
    ref = oi.int8_linear(x, qw8, sc)
    qn = ol.rms_norm(ref[:, : heads * d].reshape(m, heads, d), nq, 1e-6)
    kn = ol.rms_norm(ref[:, heads * d : (heads + kv_heads) * d].reshape(m, kv_heads, d), nk, 1e-6)
    qo, _ = ol.apply_rope(qn, kn, cos_t[pos], sin_t[pos])
    assert rel_l2(q1.cpu(), qo) < 1e-2


@pytest.mark.parametrize("m,n,k", [(300, 1000, 1024), (2048, 5120, 1024)])
@pytest.mark.parametrize("epilogue", [0, 1, 2])
def test_gemm_unaligned_output_rows(m, n, k, epilogue):
    """Output (and residual) rows whose stride is not a multiple of 8 elements take the kernels'
    element-by-element stores; the values match the aligned call bit for bit (the 128 x 128 tiling
    at 300 tokens, the 256 x 256 one at 2048)."""
    q, s = oi.quantize_int8(_bf16((n, k), seed=n + k + 5, std=0.02))
    x = _bf16((m, k), seed=m + 13)
    xd, qd, sd = x.to(DEV), q.to(DEV), s.to(DEV)
    cols = n // 2 if epilogue == 1 else n
    r = _bf16((m, n), seed=m + 14).to(DEV)

    def run(pad):
        y = torch.zeros(m, cols + pad, dtype=torch.bfloat16, device=DEV)
        rr = torch.zeros(m, n + pad, dtype=torch.bfloat16, device=DEV)
        rr[:, :n] = r
        _native.call("msa_int8_gemm", kernels._ptr(xd), m, k, k, kernels._ptr(qd), kernels._ptr(sd), n,
                     kernels._ptr(y), cols + pad, epilogue, kernels._ptr(rr) if epilogue == 2 else None,
                     n + pad if epilogue == 2 else 0, kernels._stream(y))
        return y[:, :cols].cpu()

    assert torch.equal(run(0), run(3))
