"""A feature pooled and padded at once: the gradients of both outputs reach the rows, whichever of them is there and whichever
backward runs first (the two share one search of the offsets)."""
import numpy as np
import pytest
import torch

from recis_amd import _lib
from recis_amd.nn import EmbeddingEngine, EmbeddingOption
from recis_amd.nn.modules.hashtable import HashtableRegister, filter_out_sparse_param
from recis_amd.optim import SparseAdagrad
from recis_amd.ragged import RaggedTensor

pytestmark = pytest.mark.gpu

SEQ, DIM, BATCH, KEYS = 12, 8, 300, 40


@pytest.mark.parametrize("combiner,weighted", [("mean", False), ("sum", True)])
@pytest.mark.parametrize("outputs", ["both", "apart_pool_first", "apart_tile_first", "pool", "tile"])
def test_gradients_of_both_outputs(rng, combiner, weighted, outputs):
    lens = rng.integers(6, 2 * SEQ, BATCH)
    off = torch.from_numpy(np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)).cuda()
    ids = torch.from_numpy(rng.integers(0, KEYS, int(off[-1]))).cuda()
    weight = torch.rand(len(ids), device="cuda") + 0.5 if weighted else None
    HashtableRegister().clear()
    common = dict(embedding_dim=DIM, block_size=64, shared_name="q")
    engine = EmbeddingEngine({"p": EmbeddingOption(combiner=combiner, use_weight=weighted, **common),
                              "t": EmbeddingOption(combiner="tile", combiner_kwargs={"tile_len": SEQ}, use_weight=False, **common)})
    engine.train()
    opt = SparseAdagrad(filter_out_sparse_param(engine), lr=0.1)
    rt = RaggedTensor(ids, off, weight)
    up_p = torch.rand(BATCH, DIM, device="cuda") + 0.5
    up_t = torch.rand(BATCH, SEQ * DIM, device="cuda") + 0.5
    # the gradient of every occurrence in 64 bits
    seg = torch.repeat_interleave(torch.arange(BATCH, device="cuda"), (off[1:] - off[:-1]).long())
    place = torch.arange(len(ids), device="cuda") - off[:-1].long()[seg]
    coef = weight.double() if weighted else torch.ones(len(ids), dtype=torch.float64, device="cuda")
    if combiner == "mean":
        coef = coef / (off[1:] - off[:-1]).double()[seg]
    grad = torch.zeros(KEYS, DIM, dtype=torch.float64, device="cuda")
    if outputs != "tile":
        grad.index_add_(0, ids, up_p.double()[seg] * coef[:, None])
    if outputs != "pool":
        kept = place < SEQ
        grad.index_add_(0, ids[kept], up_t.double().view(BATCH, SEQ, DIM)[seg[kept], place[kept]])
    out = engine({"p": rt, "t": rt})
    if outputs == "both":
        torch.autograd.backward([out["p"], out["t"]], [up_p, up_t])
    elif outputs == "apart_pool_first":
        out["p"].backward(up_p)
        out["t"].backward(up_t)
    elif outputs == "apart_tile_first":
        out["t"].backward(up_t)
        out["p"].backward(up_p)
    else:
        out["p" if outputs == "pool" else "t"].backward(up_p if outputs == "pool" else up_t)
    opt.step()
    opt.zero_grad()
    # the accumulator holds the squared gradient of every key's row, the keys' rows in some order: compared column by
    # column in order of size (a sum of about 700 terms in float32: 700 * 2^-24 of its size)
    (table,) = engine.hashtables().values()
    slot = table._hashtable_impl.slot_group().slot_by_name("sparse_adagrad_accum")
    accum = torch.cat(slot.kernel_blocks()[0]).double().sqrt().sort(0, descending=True).values
    want = grad.sort(0, descending=True).values
    torch.testing.assert_close(accum[:KEYS], want, rtol=1e-4, atol=1e-6)
    assert not accum[KEYS:].any()
    assert _lib.poll_device_errors() == 0


@pytest.mark.parametrize("weighted", [False, True])
@pytest.mark.parametrize("first", ["together", "pool"])
def test_gradients_of_both_outputs_of_long_segments(rng, weighted, first):
    """More than half a million ids in long segments: the pooling leaves no notes, and both backwards take their lists from
    one search of the offsets (or, when the pooled output's comes first, from one each)."""
    segments, keys = 300, 30000
    lens = rng.integers(1500, 2600, segments)
    off = torch.from_numpy(np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)).cuda()
    n = int(off[-1])
    assert n > 1 << 19
    ids = torch.from_numpy(rng.integers(0, keys, n)).cuda()
    weight = torch.rand(n, device="cuda") + 0.5 if weighted else None
    HashtableRegister().clear()
    common = dict(embedding_dim=4, block_size=4096, shared_name="q")
    engine = EmbeddingEngine({"p": EmbeddingOption(combiner="mean", use_weight=weighted, **common),
                              "t": EmbeddingOption(combiner="tile", combiner_kwargs={"tile_len": SEQ}, use_weight=False, **common)})
    engine.train()
    opt = SparseAdagrad(filter_out_sparse_param(engine), lr=0.1)
    up_p, up_t = torch.rand(segments, 4, device="cuda") + 0.5, torch.rand(segments, SEQ * 4, device="cuda") + 0.5
    seg = torch.repeat_interleave(torch.arange(segments, device="cuda"), (off[1:] - off[:-1]).long())
    place = torch.arange(n, device="cuda") - off[:-1].long()[seg]
    coef = (weight.double() if weighted else torch.ones(n, dtype=torch.float64, device="cuda")) / (off[1:] - off[:-1]).double()[seg]
    grad = torch.zeros(keys, 4, dtype=torch.float64, device="cuda").index_add_(0, ids, up_p.double()[seg] * coef[:, None])
    kept = place < SEQ
    grad.index_add_(0, ids[kept], up_t.double().view(segments, SEQ, 4)[seg[kept], place[kept]])
    rt = RaggedTensor(ids, off, weight)
    out = engine({"p": rt, "t": rt})
    if first == "together":
        torch.autograd.backward([out["p"], out["t"]], [up_p, up_t])
    else:
        out["p"].backward(up_p)
        out["t"].backward(up_t)
    opt.step()
    (table,) = engine.hashtables().values()
    held, rows = table._hashtable_impl.ids_map()
    slot = table._hashtable_impl.slot_group().slot_by_name("sparse_adagrad_accum")
    accum = torch.cat(slot.kernel_blocks()[0])[rows].double()
    # sums of about 50 terms in float32, squared
    torch.testing.assert_close(accum, grad[held] ** 2, rtol=1e-5, atol=1e-12)
    assert _lib.poll_device_errors() == 0
