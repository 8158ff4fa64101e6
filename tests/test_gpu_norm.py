"""GPU parity of RMSNorm over the row widths at which its kernels change: a wavefront per row (below
2048 and above 8192), a workgroup per row with one, two or four 16-byte pieces per thread (2048, up to
4096, up to 8192), ragged widths among them. Within rel-L2 2e-3 of the oracle: the order of the sum of
squares moves the row factor by float32 roundings, which flip bf16 roundings of single elements."""

from __future__ import annotations

import pytest
import torch
from helpers import rel_l2

from miniserve_amd import kernels
from oracle import layers as ol

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")


def _bf16(shape, seed, std=1.0):
    return (torch.randn(shape, generator=torch.Generator().manual_seed(seed)) * std).to(torch.bfloat16)


@pytest.mark.parametrize("rows,dim", [(1, 2048), (3, 2056), (5, 4096), (2, 4104), (7, 8192), (3, 8200), (9, 1024)])
def test_rmsnorm_row_widths(rows, dim):
    x, w = _bf16((rows, dim), seed=dim, std=2.0), _bf16((dim,), seed=4, std=0.1) + 1
    xd = x.to(DEV)
    out = kernels.rmsnorm(xd, w.to(DEV), 1e-6)
    assert rel_l2(out.cpu(), ol.rms_norm(x, w, 1e-6)) < 2e-3
    assert torch.equal(kernels.rmsnorm(xd, w.to(DEV), 1e-6, out=xd), out)  # in place


@pytest.mark.parametrize("dim", [1024, 2056, 4096, 8192, 8200])
def test_rmsnorm_non_finite_rows(dim):
    """An infinity (the row's factor is 0: NaN there, zeros elsewhere), a NaN, squares past float32, and
    bf16's lowest values; the rows between as ever."""
    x, w = _bf16((6, dim), seed=dim, std=2.0), _bf16((dim,), seed=4, std=0.1) + 1
    x[0, dim - 1], x[2, 3], x[3, 0] = float("-inf"), float("nan"), 3e38
    x[5] = torch.finfo(torch.bfloat16).min
    out, want = kernels.rmsnorm(x.to(DEV), w.to(DEV), 1e-6).cpu(), ol.rms_norm(x, w, 1e-6)
    assert torch.equal(out.isnan(), want.isnan()) and want[0].isnan().sum() == 1 and want[2].isnan().all()
    assert torch.equal(out[[0, 3, 5]].nan_to_num(7.0), want[[0, 3, 5]].nan_to_num(7.0))
    assert rel_l2(out[[1, 4]], want[[1, 4]]) < 2e-3


def test_rmsnorm_more_rows_than_a_launch_of_row_workgroups_holds():
    """2^24 + 3 rows of 2048 in place (69 GB): a workgroup of 256 per row would be past 2^32 work items. The
    first, middle and last rows against the same rows alone."""
    rows, dim = (1 << 24) + 3, 2048
    if torch.cuda.mem_get_info()[0] < rows * dim * 2 + (4 << 30):
        pytest.skip("needs 73 GB of free device memory")
    w = (_bf16((dim,), seed=4, std=0.1) + 1).to(DEV)
    sample = _bf16((64, dim), seed=6, std=2.0).to(DEV)
    x = torch.full((rows, dim), 0.5, dtype=torch.bfloat16, device=DEV)
    places = [0, 1 << 23, rows - 64]
    for at in places:
        x[at : at + 64] = sample
    want = kernels.rmsnorm(sample, w, 1e-6)
    kernels.rmsnorm(x, w, 1e-6, out=x)
    for at in places:
        assert rel_l2(x[at : at + 64].cpu(), want.cpu()) < 2e-3
    del x
    torch.cuda.empty_cache()
