"""Sums and row updates over the lists of a plan (recis_csr_gather_reduce, _parts, _adagrad) with hot rows, few and many entries: hot
rows go through shuffles up to half a million entries, beyond it each lane group loads its own."""
import numpy as np
import pytest
import torch

from recis_amd import _lib, ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("entries", [20_000, 500_000, 540_000])
@pytest.mark.parametrize("dim,dtype", [(16, torch.float32), (12, torch.float32), (32, torch.bfloat16), (8, torch.float32),
                                       (32, torch.float32), (15, torch.float32), (200, torch.float32)])
def test_hot_and_other_rows(rng, dim, dtype, entries):
    lens = [1, 2, 8, 9, 40, 64, 65, 2048, 2049, 5000] + [3] * ((entries - 9286) // 3)
    uniques = len(lens)
    ids = rng.permutation(np.repeat(rng.choice(10**12, uniques, replace=False), lens))
    n = len(ids)
    plan = ops.ids_unique_plan(torch.from_numpy(ids).cuda())
    rows = torch.randint(-4, 5, (n, dim), device="cuda").to(dtype)  # small whole numbers: every sum is exact in float
    src = plan.occ[:n].clone()
    coef = torch.randint(-2, 3, (n,), device="cuda").float()
    of = torch.repeat_interleave(torch.arange(uniques, device="cuda"), plan.row_start[: uniques + 1].long().diff())
    terms = rows[src.long()].double() * coef[:, None]
    want = torch.zeros(uniques, dim, dtype=torch.float64, device="cuda").index_add_(0, of, terms).float()
    assert torch.equal(ops.csr_gather_reduce(rows, plan, src, coef), want)
    plain = torch.zeros(uniques, dim, dtype=torch.float64, device="cuda").index_add_(0, of, rows[src.long()].double()).float()
    parts = [rows[: n // 3], rows[n // 3:]]
    assert torch.equal(ops.csr_gather_reduce_parts(parts, plan, src), plain)

    index = torch.randperm(uniques, device="cuda")
    slot = lambda: [(torch.rand(uniques, dim, generator=torch.Generator().manual_seed(3)) + 0.1).to(dtype).cuda()]
    w, acc, w2, acc2 = slot(), slot(), slot(), slot()
    ops.block_apply_adagrad(index, want, w, acc, 1e-2, 1e-8, uniques)
    ops.csr_gather_reduce_adagrad(rows, plan, src, coef, index, w2, acc2, 1e-2, 1e-8, uniques)
    assert torch.equal(w[0], w2[0]) and torch.equal(acc[0], acc2[0])
    assert _lib.poll_device_errors() == 0
