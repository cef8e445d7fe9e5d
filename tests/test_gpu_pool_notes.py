"""Pooling of table rows with weights, and what it notes per occurrence for the backward, against torch in 64 bits and
recis_csr_fill_lists."""
import ctypes

import numpy as np
import pytest
import torch

from recis_amd import _lib, ops

pytestmark = pytest.mark.gpu


def _p(t):
    return ctypes.c_void_p(None if t is None else t.data_ptr())


def _i(x):
    return ctypes.c_int64(x)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("weighted,mean", [(True, False), (True, True), (False, True), (False, False)])
@pytest.mark.parametrize("segments,mean_len,dim", [(300, 1, 16), (1000, 7, 24), (257, 30, 64), (129, 8, 256), (33, 400, 128),
                                                   (500, 9, 3)])
def test_pool_rows_with_notes(rng, dtype, weighted, mean, segments, mean_len, dim):
    dev = "cuda"
    lens = rng.poisson(mean_len, segments)
    lead = 5  # ids in front of the first segment and behind the last: in none
    off = torch.from_numpy(np.concatenate([[0], np.cumsum(lens)]).astype(np.int32) + lead).to(dev)
    n, rows = int(off[-1]) + lead, 200
    emb = torch.randn(rows, dim, device=dev).to(dtype)
    row_index = torch.from_numpy(rng.permutation(rows)).to(dev)
    row_index[3] = -1  # a key the table does not hold reads as zeros
    rev = torch.from_numpy(rng.integers(0, rows, n).astype(np.int32)).to(dev)
    weight = (torch.rand(n, device=dev) + 0.5).to(dtype) if weighted else None
    blocks = torch.tensor([emb.data_ptr()], dtype=torch.int64, device=dev)
    out = torch.empty(segments, dim, dtype=dtype, device=dev)
    occ = torch.empty(n, 2, dtype=torch.int32, device=dev)
    code = _lib.dtype_code(dtype)
    rc = _lib.lib().recis_segment_reduce_forward_blocks_occ(
        _p(blocks), _i(1), _i(rows), _i(0), _p(row_index), code, _p(weight), code if weighted else 0, _p(rev), 0, _p(off),
        0, _p(out), code, _i(n), _i(rows), _i(segments), _i(dim), _lib.MODES["mean" if mean else "sum"], _p(occ), _lib.stream_ptr())
    assert rc == 0
    table = emb.double()[row_index.clamp(min=0)] * (row_index >= 0).double()[:, None]
    seg = torch.repeat_interleave(torch.arange(segments, device=dev), (off[1:] - off[:-1]).long())
    coef = weight.double()[lead:n - lead] if weighted else torch.ones(n - 2 * lead, dtype=torch.float64, device=dev)
    want = torch.zeros(segments, dim, dtype=torch.float64, device=dev)
    terms = table[rev.long()[lead:n - lead]] * coef[:, None]
    want.index_add_(0, seg, terms)
    size = torch.zeros_like(want).index_add_(0, seg, terms.abs())
    if mean:
        length = (off[1:] - off[:-1]).clamp(min=1).double()[:, None]
        want, size = want / length, size / length
    # a sum of L terms in float32: (L + 1) * 2^-24 of the terms' size, and one rounding to the table's type
    bound = (int(lens.max()) + 2) * 2.0 ** -24 * size + (2.0 ** -8 if dtype == torch.bfloat16 else 0) * want.abs() + 1e-30
    assert bool(((out.double() - want).abs() <= bound).all())

    order = torch.from_numpy(rng.permutation(n).astype(np.int32)).to(dev)
    lists = []
    for notes in (True, False):
        src = torch.empty(n, dtype=torch.int32, device=dev)
        c = torch.empty(n, dtype=torch.float32, device=dev) if weighted or mean else None
        if notes:
            rc = _lib.lib().recis_csr_lists_from_occ(_p(order), _i(n), _p(occ), _p(off), 0, _i(segments), _p(src), _p(c),
                                                     _lib.stream_ptr())
        else:
            rc = _lib.lib().recis_csr_fill_lists(_p(order), _i(n), _p(off), 0, _i(segments), _p(weight), code if weighted else 0,
                                                 int(mean), _p(src), _p(c), None, None, _i(0), None, _lib.stream_ptr())
        assert rc == 0
        lists.append((src, c))
    assert torch.equal(lists[0][0], lists[1][0])
    if lists[0][1] is not None:
        assert torch.equal(lists[0][1], lists[1][1])
    assert _lib.poll_device_errors() == 0


@pytest.mark.parametrize("off64", [0, 1])
@pytest.mark.parametrize("weighted,mean", [(False, False), (True, True)])
@pytest.mark.parametrize("offsets", [[0, 4, 99, 8], [0, 4, 8, -3, 8], [-2, 3, 8], [0, 3, 3, 8], [2, 5, 7]])
def test_occurrences_of_bad_segments_have_no_notes(rng, offsets, weighted, mean, off64):
    """Segments with bad offsets note nothing: their occurrences, which added nothing to any output, take no
    gradient, whatever the buffer of the notes held before."""
    n, dim, rows, S = 8, 4, 5, len(offsets) - 1
    dev = "cuda"
    off = torch.tensor(offsets, dtype=torch.int64 if off64 else torch.int32, device=dev)
    emb = torch.randn(rows, dim, device=dev)
    row_index = torch.arange(rows, device=dev)
    rev = torch.from_numpy(rng.integers(0, rows, n).astype(np.int32)).to(dev)
    weight = torch.rand(n, device=dev) + 0.5 if weighted else None
    blocks = torch.tensor([emb.data_ptr()], dtype=torch.int64, device=dev)
    out = torch.empty(S, dim, device=dev)
    order = torch.from_numpy(rng.permutation(n).astype(np.int32)).to(dev)
    want_src, want_coef = np.full(n, -1), np.zeros(n)
    for s, (a, b) in enumerate(zip(offsets[:-1], offsets[1:])):
        if 0 <= a <= b <= n:
            want_src[a:b] = s
            want_coef[a:b] = (weight[a:b].cpu().numpy() if weighted else 1.0) / np.float32((b - a) if mean else 1)
    for junk in (0, 1, S - 1, S, -1, 1 << 30):
        occ = torch.empty(n, 2, dtype=torch.int32, device=dev)
        occ[:, 0] = junk
        occ[:, 1] = torch.tensor([7.5], device=dev).view(torch.int32)
        assert _lib.lib().recis_segment_reduce_forward_blocks_occ(
            _p(blocks), _i(1), _i(rows), _i(0), _p(row_index), 0, _p(weight), 0, _p(rev), 0, _p(off), off64, _p(out), 0, _i(n),
            _i(rows), _i(S), _i(dim), _lib.MODES["mean" if mean else "sum"], _p(occ), _lib.stream_ptr()) == 0
        src = torch.full((n,), 123, dtype=torch.int32, device=dev)
        coef = torch.full((n,), 123.0, device=dev)
        assert _lib.lib().recis_csr_lists_from_occ(_p(order), _i(n), _p(occ), _p(off), off64, _i(S), _p(src), _p(coef),
                                                   _lib.stream_ptr()) == 0
        at = order.cpu().numpy()
        assert (src.cpu().numpy() == want_src[at]).all(), junk
        np.testing.assert_allclose(coef.cpu().numpy(), want_coef[at], rtol=2.0 ** -23)  # one division in float32
    _lib.poll_device_errors()


@pytest.mark.parametrize("n", [1, 2, 256, 1023, 70001])
@pytest.mark.parametrize("kind", ["one in each", "first", "last", "random", "off by one"])
@pytest.mark.parametrize("weighted,mean", [(False, False), (False, True), (True, True)])
def test_lists_of_as_many_segments_as_ids(rng, n, kind, weighted, mean):
    off = np.arange(n + 1)
    if kind == "first":
        off[1:-1] += 1 if n > 1 else 0
    elif kind == "last":
        off[-2:] = n if n > 1 else off[-2:]
    elif kind == "random":
        off[1:-1] = np.sort(rng.integers(0, n + 1, n - 1))
    elif kind == "off by one":  # id 0 in no segment
        off[:-1] += 1
    ids = rng.integers(0, max(1, n // 3), n)
    plan = ops.ids_unique_plan(torch.from_numpy(ids).cuda())
    w = (rng.random(n) + 0.5).astype(np.float32)
    src, coef = plan.src_coef_for_pool(torch.from_numpy(off.astype(np.int32)).cuda(),
                                       torch.from_numpy(w).cuda() if weighted else None, mean)
    at = plan.occ.cpu().numpy()
    want = np.searchsorted(off, np.arange(n), side="right") - 1
    inside = (np.arange(n) >= off[0]) & (np.arange(n) < off[-1])
    c = (w if weighted else np.ones(n, np.float32)) / (np.maximum(np.diff(off)[want], 1) if mean else 1)
    assert (src.cpu().numpy() == np.where(inside, want, -1)[at]).all()
    if weighted or mean:
        np.testing.assert_allclose(coef.cpu().numpy(), np.where(inside, c, 0)[at], rtol=2.0 ** -23)
    assert _lib.poll_device_errors() == 0
