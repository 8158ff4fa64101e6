"""GPU parity of the GEMM shapes that split K in two on 256 x 128 tiles because their tiles leave half the
chip idle (96 to 128 tiles) against the CPU oracle: the edges of that range, ragged tokens and rows,
the shapes just outside it, with and without a workspace. Bars as for the other GEMMs: rel-L2 1e-2 of
the oracle, 4e-3 (one bf16 rounding) of float64, the residual exact on the kernel's own product."""

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


@pytest.mark.parametrize("m,n,k,split", [
    (768, 4096, 2048, True),  # 96 tiles
    (530, 4000, 2048, True),  # ragged both ways, 96 tiles
    (1024, 4096, 2048, True),  # 128 tiles
    (1500, 2048, 4096, True),  # 96 tiles, the plain linear split too
    (1020, 3968, 2112, False),  # 124 tiles, K steps that do not halve
    (1025, 4096, 2048, False),  # 160 tiles
    (768, 4096, 1024, False),  # halves of 512
    (1300, 2560, 2048, False),  # 120 tiles, of which four XCDs would take 36 workgroups
    (1536, 2048, 2048, True),  # 96 tiles, 24 workgroups on each
])
def test_gemm_mid_splits(m, n, k, split):
    q, s = oi.quantize_int8(_bf16((n, k), seed=n + k, std=0.02))
    x, r, w = _bf16((m, k), seed=m), _bf16((m, n), seed=m + 1), _bf16((n,), seed=3, std=0.1) + 1
    xd, qd, sd = x.to(DEV), q.to(DEV), s.to(DEV)
    assert (_native.query("msa_int8_linear_add_rmsnorm_workspace_size", m, n, k) == 2 * m * n * 4) is split
    y = kernels.int8_linear(xd, qd, sd)
    assert torch.equal(y, kernels.int8_linear(xd, qd, sd))
    exact = x.double() @ oi.dequantize(q, s, torch.bfloat16).double().T
    assert rel_l2(y.cpu(), oi.int8_linear(x, q, s)) < 1e-2
    assert rel_l2(y.cpu(), exact) < 4e-3
    y2 = torch.empty_like(y)
    _native.call("msa_int8_gemm", kernels._ptr(xd), m, k, k, kernels._ptr(qd), kernels._ptr(sd), n, kernels._ptr(y2),
                 n, 0, None, 0, kernels._stream(y2))  # no workspace: never split
    assert rel_l2(y2.cpu(), exact) < 4e-3
    acc = r.to(DEV)
    kernels.int8_linear(xd, qd, sd, kernels.EPI_RESIDUAL, residual=acc, out=acc)
    assert torch.equal(acc.cpu(), (r.float() + y.cpu().float()).to(torch.bfloat16))
    res = r.to(DEV)
    out = kernels.int8_linear_add_rmsnorm(xd, qd, sd, res, w.to(DEV), 1e-6)
    # (the plain linear splits only from k = 4096 on: another order of the float32 sums flips single
    # bf16 roundings, 2^-9 of a value each)
    assert torch.equal(res, acc) if k >= 4096 or not split else rel_l2(res.cpu(), acc.cpu()) < 2e-3
    assert rel_l2(out.cpu(), ol.rms_norm(res.cpu(), w, 1e-6)) < 2e-3
