"""The gather-reduce with two inputs on short lists: the lists of a wave are worked side by side, one, two or four rows of
each at a time as the longest of them asks, and a key's table row is asked for before its gradient is summed."""
import ctypes
import types

import numpy as np
import pytest
import torch

from recis_amd import _lib, ops

pytestmark = pytest.mark.gpu

LENGTHS = {"ones": [1], "twos": [1, 2], "threes": [1, 3, 2], "short": [1, 2, 4, 5, 8], "mixed": [1, 8, 9, 2, 64, 3, 65, 40, 1, 2100]}


@pytest.mark.parametrize("blocks", [1, 3])
@pytest.mark.parametrize("dim,dtype", [(128, torch.bfloat16), (72, torch.bfloat16), (32, torch.bfloat16), (16, torch.float32), (64, torch.float32), (36, torch.float32),
                                       (1030, torch.float32)])
@pytest.mark.parametrize("lengths", sorted(LENGTHS))
def test_short_lists_of_two_inputs(rng, lengths, dim, dtype, blocks):
    uniques = 40 if dim > 512 else 150
    lens = [LENGTHS[lengths][u % len(LENGTHS[lengths])] for u in range(uniques)]
    ids = rng.permutation(np.repeat(rng.choice(10**9, uniques, replace=False), lens))
    n = len(ids)
    plan = ops.ids_unique_plan(torch.from_numpy(ids).cuda())
    occ = plan.occ[:n].cpu().numpy()
    segments = max(1, n // 7)
    seg = rng.integers(0, segments, size=n)
    src1, src2 = seg[occ].astype(np.int32), occ.astype(np.int32)
    src2[rng.random(n) < 0.1] = -1  # entries that read nothing
    coef = rng.random(n).astype(np.float32)
    rows1 = torch.randn(segments, dim).to(dtype)
    rows2 = torch.randn(n, dim).to(dtype)
    lost = int(occ[n // 2])  # one row that is not finite reaches its own id only
    rows2[lost] = float("inf")
    half = n // 2
    first = (rows1.cuda(), torch.from_numpy(src1).cuda(), torch.from_numpy(coef).cuda())
    second = ([rows2[:half].cuda(), rows2[half:].cuda()], torch.from_numpy(src2).cuda(), None)
    got = ops.csr_gather_reduce2(plan, first, second).cpu().numpy()

    of = np.repeat(np.arange(uniques), np.diff(plan.row_start.cpu().numpy()[: uniques + 1]))
    want, size = np.zeros((uniques, dim)), np.zeros((uniques, dim))
    r1, r2 = rows1.double().numpy(), rows2.double().numpy()
    terms = [(coef[:, None] * r1[src1], of), (r2[src2[src2 >= 0]], of[src2 >= 0])]
    for t, o in terms:
        np.add.at(want, o, t)
        np.add.at(size, o, np.abs(t))
    # a sum of k products in float: at most k + 1 roundings of relative size 2^-24 on every partial sum
    bound = (2 * np.array([np.count_nonzero(of == u) for u in range(uniques)])[:, None] + 2) * 2.0**-24 * size
    ok = np.isfinite(want)
    assert np.all(np.abs(got - want)[ok] <= bound[ok]) and not np.isfinite(got[~ok]).any()

    # the update at once: the bits of the sum in float and the stand-alone row kernel
    held = uniques * 2
    size_of_block = -(-held // blocks)
    index = torch.from_numpy(rng.choice(held, uniques, replace=False)).cuda()
    index[uniques // 3] = -1  # a key the table does not hold
    def slot(positive):
        t = torch.randn(blocks * size_of_block, dim, generator=torch.Generator().manual_seed(3))
        t = (t.square() + 0.1 if positive else t).to(dtype)
        return [b.cuda() for b in torch.split(t, size_of_block)]
    w, acc, w2, acc2 = slot(False), slot(True), slot(False), slot(True)
    total = ops.csr_gather_reduce2(plan, first, second)
    total[uniques // 3] = 0
    known = torch.arange(uniques, device="cuda") != uniques // 3
    ops.block_apply_adagrad(index[known], total[known], w, acc, 1e-2, 1e-8, size_of_block)
    ops.csr_gather_reduce2_adagrad(plan, first, second, index, w2, acc2, 1e-2, 1e-8, size_of_block)
    for a, b in zip(w + acc, w2 + acc2):
        assert torch.equal(torch.nan_to_num(a.float()), torch.nan_to_num(b.float()))
    s0, s1, m0, m1 = slot(False), slot(True), slot(False), slot(True)
    powers = [torch.full((1,), v, dtype=torch.float64, device="cuda") for v in (0.9, 0.999, 0.9, 0.999)]
    ops.block_apply_adamw(index[known], total[known], w, powers[0], powers[1], None, s0, s1,
                          1e-2, 0.9, 0.999, 0.99, 1e-8, size_of_block)
    ops.csr_gather_reduce2_adamw(plan, first, second, index, w2, powers[2], powers[3], m0, m1, 1e-2, 0.9, 0.999, 0.99, 1e-8,
                                 size_of_block)
    for a, b in zip(w + s0 + s1, w2 + m0 + m1):
        assert torch.equal(torch.nan_to_num(a.float()), torch.nan_to_num(b.float()))
    assert _lib.poll_device_errors() == 0


@pytest.mark.parametrize("blocks", [1, 3])
@pytest.mark.parametrize("dim,dtype", [(128, torch.float32), (132, torch.float32), (256, torch.float32), (1030, torch.float32),
                                       (33, torch.float32), (264, torch.bfloat16)])
def test_lists_of_any_length_without_work_items(rng, dim, dtype, blocks):
    """hot_cap == 0: no list is too long for the row kernel, also where a row takes all lanes of a wave."""
    lens = [64, 65, 200, 1, 66, 100, 130, 8, 9]
    uniques = len(lens)
    ids = rng.permutation(np.repeat(rng.choice(10**9, uniques, replace=False), lens))
    n = len(ids)
    made = ops.ids_unique_plan(torch.from_numpy(ids).cuda())
    plan = types.SimpleNamespace(U=uniques, row_start=made.row_start, hot_items=None, hot_cap=0, counts=made.counts)
    occ = made.occ[:n].cpu().numpy()
    # small whole numbers: every sum is exact in float
    rows1, rows2 = (torch.randint(-8, 9, (n, dim)).to(dtype) for _ in range(2))
    src1 = rng.permutation(n).astype(np.int32)
    coef = rng.integers(-3, 4, size=n).astype(np.float32)
    first = (rows1.cuda(), torch.from_numpy(src1).cuda(), torch.from_numpy(coef).cuda())
    second = (rows2.cuda(), torch.from_numpy(occ).cuda(), None)
    of = np.repeat(np.arange(uniques), np.diff(made.row_start.cpu().numpy()[: uniques + 1]))
    want = np.zeros((uniques, dim))
    np.add.at(want, of, coef[:, None] * rows1.double().numpy()[src1] + rows2.double().numpy()[occ])
    np.testing.assert_array_equal(ops.csr_gather_reduce2(plan, first, second).cpu().numpy(), want)

    size_of_block = uniques
    index = torch.from_numpy(rng.permutation(blocks * size_of_block)[:uniques]).cuda()
    total = torch.from_numpy(want).float().cuda()
    def slot():
        t = (torch.rand(blocks * size_of_block, dim, generator=torch.Generator().manual_seed(3)) + 0.1).to(dtype)
        return [b.cuda() for b in torch.split(t, size_of_block)]
    w, acc, w2, acc2 = slot(), slot(), slot(), slot()
    ops.block_apply_adagrad(index, total, w, acc, 1e-2, 1e-8, size_of_block)
    ops.csr_gather_reduce2_adagrad(plan, first, second, index, w2, acc2, 1e-2, 1e-8, size_of_block)
    for a, b in zip(w + acc, w2 + acc2):
        assert torch.equal(a, b)
    s0, s1, m0, m1 = slot(), slot(), slot(), slot()
    powers = [torch.full((1,), v, dtype=torch.float64, device="cuda") for v in (0.9, 0.999, 0.9, 0.999)]
    ops.block_apply_adamw(index, total, w, powers[0], powers[1], None, s0, s1, 1e-2, 0.9, 0.999, 0.99, 1e-8, size_of_block)
    ops.csr_gather_reduce2_adamw(plan, first, second, index, w2, powers[2], powers[3], m0, m1, 1e-2, 0.9, 0.999, 0.99, 1e-8,
                                 size_of_block)
    for a, b in zip(w + s0 + s1, w2 + m0 + m1):
        assert torch.equal(a, b)
    assert _lib.poll_device_errors() == 0


def test_rows_past_the_count_are_not_asked_for(rng):
    """U may be a bound (the number of ids): row_index need not hold more rows than there are unique ids."""
    from recis_amd._lib import check, dtype_code, i64, lib, ptr, stream_ptr

    dim, uniques = 64, 300
    ids = torch.from_numpy(rng.permutation(np.repeat(rng.choice(10**9, uniques, replace=False), 9))).cuda()
    n = ids.numel()
    plan = ops.ids_unique_plan(ids)
    first = (torch.randn(n, dim, device="cuda"), plan.occ[:n], None)
    second = (torch.randn(n, dim, device="cuda"), plan.occ[:n].flip(0), None)
    index = torch.randperm(uniques, device="cuda")
    slot = lambda: [torch.rand(uniques, dim, generator=torch.Generator().manual_seed(3)).cuda()]
    w, acc, w2, acc2 = slot(), slot(), slot(), slot()
    ops.csr_gather_reduce2_adagrad(plan, first, second, index, w, acc, 1e-2, 1e-8, uniques)
    head, _, dev, keep = ops._two_inputs(plan, first, second)
    check(lib().recis_csr_gather_reduce2_adagrad(
        *head, i64(n), i64(dim), ptr(index), ptr(ops.block_ptr_table(w2)), ptr(ops.block_ptr_table(acc2)), i64(1), i64(uniques),
        i64(0), dtype_code(torch.float32), ctypes.c_double(1e-2), ctypes.c_double(1e-8), stream_ptr(dev)))
    assert torch.equal(w[0], w2[0]) and torch.equal(acc[0], acc2[0])
    assert _lib.poll_device_errors() == 0
