"""recis_collect_rows (strided parts laid end to end in one array) against torch.cat, and the training step whose outputs'
gradients are column slices against the one that gets them as dense arrays."""
import ctypes

import numpy as np
import pytest
import torch

from recis_amd import _lib, ops
from recis_amd.nn import EmbeddingEngine, EmbeddingOption
from recis_amd.nn.modules.hashtable import HashtableRegister, filter_out_sparse_param
from recis_amd.optim import SparseAdagrad, SparseAdam

pytestmark = pytest.mark.gpu


def _collect(parts, counts, dim, dtype):
    rows = sum(counts)
    out = torch.full((rows, dim), 7, dtype=dtype, device="cuda")
    base = (ctypes.c_void_p * len(parts))(*[None if p is None else p.data_ptr() for p in parts])
    stride = (ctypes.c_int64 * len(parts))(*[0 if p is None else p.stride(0) * p.element_size() for p in parts])
    rc = _lib.lib().recis_collect_rows(base, stride, (ctypes.c_int64 * len(parts))(*counts), ctypes.c_int64(len(parts)),
                                       ctypes.c_int64(dim * out.element_size()), out.element_size(),
                                       ctypes.c_void_p(out.data_ptr()), _lib.stream_ptr())
    return rc, out


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("dim", [1, 3, 10, 16, 24, 130, 1000])
@pytest.mark.parametrize("n_parts,alike", [(1, True), (2, True), (2, False), (39, True), (64, False), (65, True)])
def test_collect_rows(rng, dtype, dim, n_parts, alike):
    counts = [1037 if n_parts < 3 else 37] * n_parts if alike else [int(c) for c in rng.integers(0, 90, n_parts)]
    wide = torch.randn(max(max(counts), 1), n_parts * dim + 1, device="cuda").to(dtype)
    parts = [wide[:c, f * dim + (f % 2):][:, :dim] for f, c in enumerate(counts)]
    if n_parts > 2:
        parts[1] = None                                             # no gradient reached it
        parts[2] = torch.randn(1, dim, device="cuda").to(dtype).expand(counts[2], dim)  # one row over and over
    flat = torch.cat([torch.zeros(c, dim, device="cuda", dtype=dtype) if p is None else p for p, c in zip(parts, counts)])
    rc, out = _collect(parts, counts, dim, dtype)
    assert rc == 0 and torch.equal(out, flat)
    assert _lib.poll_device_errors() == 0


@pytest.mark.parametrize("optim", [SparseAdam, SparseAdagrad])
@pytest.mark.parametrize("dim", [4, 16, 64])
def test_step_with_column_slices_matches_dense_gradients(rng, optim, dim):
    """The same step with the outputs' gradients as column slices of one array (collected) and as one dense
    array after the other (read in place): sums of at most 700 terms in two orders, 700 * 2^-24 of the terms' size."""
    names = ["a", "b", "c"]
    ids = {n: torch.from_numpy(rng.integers(0, 3 + 400 * k, (700, 1))).cuda() for k, n in enumerate(names)}
    up = torch.rand(700, 3 * dim, device="cuda") + 0.5
    rows = []
    for sliced in (True, False):
        HashtableRegister().clear()
        torch.manual_seed(0)
        engine = EmbeddingEngine({n: EmbeddingOption(embedding_dim=dim, block_size=512, shared_name=n, combiner="sum",
                                                     use_weight=False) for n in names})
        engine.train()
        opt = optim(filter_out_sparse_param(engine), lr=0.1)
        for _ in range(2):
            out = engine(ids)
            if sliced:
                torch.cat([out[n] for n in names], dim=1).backward(up)
            else:
                torch.autograd.backward([out[n] for n in names], list(torch.stack(up.split(dim, 1))))
            opt.step()
            opt.zero_grad()
        with torch.no_grad():
            out = engine.eval()(ids)
        rows.append(torch.cat([out[n] for n in names], dim=1))
    torch.testing.assert_close(rows[0], rows[1], rtol=1e-4, atol=1e-5)
    assert _lib.poll_device_errors() == 0


@pytest.mark.parametrize("dtype,dim", [(torch.float32, 4), (torch.float32, 16), (torch.bfloat16, 10), (torch.float32, 300)])
@pytest.mark.parametrize("n_parts,count", [(1, 8191), (2, 33333), (3, 65536), (17, 9001)])
def test_collect_rows_of_few_large_parts(dtype, dim, n_parts, count):
    """Few parts: a workgroup takes more rows of each, up to what its lane groups have in flight."""
    wide = torch.randn(count, n_parts * dim, device="cuda").to(dtype)
    parts = list(wide.split(dim, 1))
    rc, out = _collect(parts, [count] * n_parts, dim, dtype)
    assert rc == 0 and torch.equal(out, torch.cat(parts))


@pytest.mark.parametrize("columns,rows_each,dim,extra,dtype", [
    (1, 1, 4, 0, torch.float32), (3, 1, 16, 0, torch.float32), (2, 7, 10, 3, torch.bfloat16), (39, 1000, 16, 0, torch.float32),
    (5, 4096, 4, 4, torch.bfloat16), (7, 65537, 1, 1, torch.float32), (3, 333, 64, 0, torch.float16), (2, 100, 600, 8, torch.float32)])
def test_sums_over_column_slices(rng, columns, rows_each, dim, extra, dtype):
    """recis_csr_gather_reduce_grid against sums of whole numbers, which no order of the additions rounds: the division by the rows of
    a column, lists of every length, entries that read nothing."""
    n = columns * rows_each
    ids = np.where(rng.random(n) < 0.5, rng.integers(0, max(1, n // 3), size=n), rng.integers(0, 3, size=n))
    plan = ops.ids_unique_plan(torch.from_numpy(ids).cuda())
    wide = torch.from_numpy(rng.integers(-3, 4, size=(rows_each, columns * dim + extra)).astype(np.float32)).to(dtype)
    src = plan.occ[:n].cpu().numpy().copy()
    src[rng.random(n) < 0.1] = -1
    where = torch.from_numpy(src).cuda()
    on = wide.cuda()
    out = torch.full((plan.U, dim), 7.0, device="cuda")
    i64 = ctypes.c_int64
    _lib.check(_lib.lib().recis_csr_gather_reduce_grid(
        _lib.ptr(on), _lib.dtype_code(dtype), i64(columns), i64(rows_each), i64(dim), i64(on.stride(0)), _lib.ptr(where),
        _lib.ptr(plan.row_start), _lib.ptr(plan.hot_items), i64(plan.hot_cap), _lib.ptr(plan.counts), _lib.ptr(out), i64(plan.U),
        i64(dim), _lib.stream_ptr(on.device)))
    rows = wide.float().numpy()[:, : columns * dim].reshape(rows_each, columns, dim).transpose(1, 0, 2).reshape(n, dim)
    want = np.zeros((plan.U, dim), np.float32)
    of = np.repeat(np.arange(plan.U), np.diff(plan.row_start.cpu().numpy()[: plan.U + 1]))
    np.add.at(want, of[src >= 0], rows[src[src >= 0]])
    np.testing.assert_array_equal(out.cpu().numpy(), want)
    assert _lib.poll_device_errors() == 0


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("form", ["slices", "gap", "reversed", "few"])
def test_gradients_of_concatenated_columns(rng, dtype, form):
    """A step whose gradients are column slices of one array against the same step with an array per column; whole
    numbers, so that sums do not depend on the order. Slices that are not side by side, or few, go the general way."""
    batch, columns, dim = (70_001, 15, 4) if form != "few" else (1000, 15, 4)
    data = {"c%d" % k: torch.from_numpy(rng.integers(0, 10 ** (1 + k % 5), size=(batch, 1))).cuda() for k in range(columns)}
    wide = torch.from_numpy(rng.integers(-2, 3, size=(batch, 2 * columns * dim)).astype(np.float32)).cuda().to(dtype)
    step = 2 * dim if form == "gap" else dim
    ups = [wide[:, k * step: k * step + dim] for k in range(columns)]
    if form == "reversed":
        ups = ups[::-1]
    tables = []
    for sliced in (True, False):
        HashtableRegister().clear()
        engine = EmbeddingEngine({n: EmbeddingOption(embedding_dim=dim, dtype=dtype, shared_name=n, combiner="sum",
                                                     use_weight=False, reserve_rows=1 << 17) for n in data})
        engine.train()
        opt = SparseAdagrad(filter_out_sparse_param(engine), lr=0.5)
        for turn in range(2):  # the second adds to rows that are not zero
            out = engine(data)
            grads = [u.clone() if not sliced else u for u in ups]
            torch.autograd.backward([out[n] for n in data], grads)
            if sliced and turn == 0:
                keep, _ = wide.clone(), wide.fill_(float("nan"))  # the caller's buffer is the caller's again
                opt.step()
                wide.copy_(keep)
            else:
                opt.step()
            opt.zero_grad()
        (table,) = engine.hashtables().values()
        impl = table._hashtable_impl
        ids, index = impl.ids_map()
        order = ids.argsort()
        tables.append((ids[order], [torch.cat(s.values())[index[order]] for s in impl.slot_group().slots()]))
    (ids_a, a), (ids_b, b) = tables
    assert torch.equal(ids_a, ids_b) and len(a) == len(b)
    for x, y in zip(a, b):
        assert torch.equal(x, y)
    assert _lib.poll_device_errors() == 0
