"""recis_collect_rows (strided parts laid end to end in one array) against torch.cat, and the training step whose outputs'
gradients are column slices against the one that gets them as dense arrays."""
import ctypes

import numpy as np
import pytest
import torch

from recis_amd import _lib
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
