"""The padded gather with its rows in a table's blocks against recis_ragged_tile over a dense copy of the rows (bit for bit)."""
import ctypes

import numpy as np
import pytest
import torch

from recis_amd import _lib

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("dim,pitch", [(1, 0), (10, 0), (24, 32), (128, 0), (300, 0)])
@pytest.mark.parametrize("batch,seq", [([5], [1]), ([33, 7], [20, 100]), ([64, 1, 3], [17, 0, 300])])
def test_tile_from_blocks(rng, dtype, dim, pitch, batch, seq):
    dev, n_blocks, block_rows, unique = "cuda", 3, 50, 90
    lens = np.concatenate([rng.integers(0, 2 * s + 2, b) for b, s in zip(batch, seq)])
    off = torch.from_numpy(np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)).to(dev)
    n = int(off[-1])
    value = torch.from_numpy(rng.integers(0, unique, max(n, 1)).astype(np.int32)).to(dev)
    width = pitch or dim
    blocks = [torch.randn(block_rows, width, device=dev).to(dtype) for _ in range(n_blocks)]
    row_index = torch.from_numpy(rng.permutation(n_blocks * block_rows)[:unique]).to(dev)
    row_index[[1, 5]] = -1
    dense = torch.cat(blocks)[row_index.clamp(min=0), :dim] * (row_index >= 0)[:, None]
    dense = dense.to(dtype).contiguous()
    table = torch.tensor([b.data_ptr() for b in blocks], dtype=torch.int64, device=dev)
    rows = sum(b * s for b, s in zip(batch, seq))
    got, want = (torch.full((rows, dim), 3, dtype=dtype, device=dev) for _ in range(2))

    def c64(x):
        return ctypes.c_int64(x)

    def vp(t):
        return ctypes.c_void_p(t.data_ptr())

    cb, cs = (ctypes.c_int64 * len(batch))(*batch), (ctypes.c_int64 * len(seq))(*seq)
    size, code = got.element_size(), _lib.dtype_code(dtype)
    assert _lib.lib().recis_ragged_tile_blocks(cb, cs, c64(len(batch)), vp(value), 0, c64(n), vp(off), 0, vp(table),
                                               c64(n_blocks), c64(block_rows), c64(pitch * size), vp(row_index), c64(unique),
                                               code, vp(got), c64(dim), _lib.stream_ptr()) == 0
    assert _lib.lib().recis_ragged_tile(cb, cs, c64(len(batch)), vp(value), 0, c64(n), vp(off), 0, vp(dense), c64(unique), code,
                                        vp(want), c64(dim), _lib.stream_ptr()) == 0
    assert torch.equal(got, want)
    assert _lib.poll_device_errors() == 0
