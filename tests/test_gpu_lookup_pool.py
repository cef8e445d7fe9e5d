"""Read-only lookup and pooling in one pass (recis_lookup_pool_readonly) against a float64 restatement: the map as a
dict, the rows looked up one by one, the sum / mean per segment."""
import numpy as np
import pytest
import torch

from recis_amd import _lib, ops
from recis_amd.nn import DynamicEmbedding, EmbeddingEngine, EmbeddingOption, HashTable
from recis_amd.nn.modules.hashtable import HashtableRegister, filter_out_sparse_param
from recis_amd.ragged import RaggedTensor

pytestmark = pytest.mark.gpu

TAG = 52


def _table(D, dtype, known, block_size, rng):
    """(HashtableImpl with rows for `known`, key -> float64 row)."""
    HashtableRegister().clear()
    ht = HashTable([D], block_size=block_size, dtype=dtype, name="pool_table")
    rows = torch.from_numpy(rng.standard_normal((len(known), D)).astype(np.float32)).to(dtype)
    ht.insert(torch.from_numpy(known).cuda(), rows.cuda())
    return ht, {int(k): r for k, r in zip(known, rows.double().numpy())}


def _feature(rng, kind, n_seg, pool):
    """(values, offsets | None, weight | None, per-segment (ids, weights))."""
    if kind in ("column", "wide"):
        width = 1 if kind == "column" else 3
        ids = rng.choice(pool, size=(n_seg, width))
        return ids if width > 1 else ids[:, 0], None, None, [(r, np.ones(width)) for r in ids]
    longest = {"short": 5, "long": 60, "huge": 3}[kind]
    lens = rng.integers(0, longest, size=n_seg)
    if kind == "huge" and n_seg:  # more ids than a workgroup keeps the rows of at a time, twice in one tile
        lens[n_seg // 2] = 2500
        lens[-1] = 1025
    off = np.concatenate([[0], np.cumsum(lens)])
    ids = rng.choice(pool, size=off[-1])
    w = rng.random(off[-1]).astype(np.float32) + 0.25
    return ids, off, w, [(ids[a:b], w[a:b]) for a, b in zip(off[:-1], off[1:])]


@pytest.mark.parametrize("mean", [False, True])
@pytest.mark.parametrize("D,dtype,weighted,tagged,kinds", [
    (16, torch.float32, False, True, ["column", "short", "column", "wide"]),
    (16, torch.float32, True, True, ["short", "huge", "long"]),
    (1, torch.float32, False, False, ["huge"]),
    (24, torch.float32, True, False, ["long"]),
    (128, torch.bfloat16, False, True, ["huge", "column"]),
    (10, torch.bfloat16, True, True, ["short", "column", "long"]),
    (100, torch.float16, False, True, ["wide", "long"]),
    (600, torch.float32, False, False, ["huge"]),
    (8, torch.float32, False, True, ["column"] * 70),  # more features than one launch takes
    (8, torch.float32, False, True, ["column", "long"] * 35),  # the ragged ones go first, over both launches
])
@pytest.mark.parametrize("n_seg", [1, 65, 3000])
def test_lookup_pool_matches_float64(rng, D, dtype, weighted, tagged, kinds, n_seg, mean):
    pool = rng.integers(0, 1 << 40, size=max(50, n_seg))
    known = np.unique(pool)[::2]  # half of the ids are unknown and read as zeros
    tags = list(range(3, 3 + len(kinds))) if tagged else None
    coded = np.concatenate([known | (t << TAG) for t in tags]) if tagged else known
    ht, rows = _table(D, dtype, coded, 64, rng)  # many small blocks
    feats = [_feature(rng, k, n_seg, pool) for k in kinds]
    if not tagged:
        assert len(feats) == 1
    values = [torch.from_numpy(f[0]).cuda() for f in feats]
    offs = [None if f[1] is None else torch.from_numpy(f[1].astype(np.int32 if i % 2 else np.int64)).cuda()
            for i, f in enumerate(feats)]
    ws = [None if f[2] is None or not weighted else torch.from_numpy(f[2]).cuda() for f in feats]
    parts = ht._hashtable_impl.lookup_pool_readonly(values, offs, ws, tags, mean)
    n_ids, n_segs = sum(v.numel() for v in values), n_seg * len(feats)
    by_length = n_ids > 5 * (n_segs + 1)
    # float32 sums of k terms: k rounding steps of 2^-24 of the summed magnitude; one rounding of the result to the row
    # type (float16: below 2^-14 its values lie 2^-24 apart)
    eps = {torch.float32: 2.0 ** -24, torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11}[dtype]
    tiny = 2.0 ** -25 if dtype == torch.float16 else 1e-30
    zero = np.zeros(D)
    for f, part, w, k in zip(feats, parts, ws, range(len(feats))):
        got = part.double().cpu().numpy()
        assert got.shape == (n_seg, D)
        for s, (ids, wt) in enumerate(f[3]):
            wt = torch.from_numpy(np.asarray(wt, np.float32)).to(dtype).double().numpy() if w is not None else np.ones(len(ids))
            x = np.array([rows.get(int(i) | ((tags[k] << TAG) if tagged else 0), zero) for i in ids]).reshape(len(ids), D)
            exp, mag = wt @ x, np.abs(wt) @ np.abs(x)
            if mean and len(ids):
                div = len(ids) if by_length else wt.sum()
                exp, mag = exp / div, mag / div
            assert np.all(np.abs(got[s] - exp) <= eps * np.abs(exp) + (len(ids) + 4) * 2.0 ** -24 * mag + tiny), (k, s)
    assert _lib.poll_device_errors() == 0


def test_evaluation_forward_equals_the_training_rows(rng):
    """EmbeddingEngine in evaluation mode (one pass) against training mode (plan, expansion, pooling) on the same table."""
    HashtableRegister().clear()
    names = ["a", "b", "c", "d"]
    eng = EmbeddingEngine({n: EmbeddingOption(embedding_dim=16, shared_name=n, combiner="sum", use_weight=n == "c")
                           for n in names})
    lens = rng.integers(0, 9, size=500)
    off = torch.from_numpy(np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)).cuda()
    n = int(off[-1])
    ids = lambda k: torch.from_numpy(rng.integers(0, 300, size=k)).cuda()
    x = {"a": ids(500).view(-1, 1), "b": RaggedTensor(ids(n), off),
         "c": RaggedTensor(ids(n), off, torch.rand(n, device="cuda")), "d": ids(1000).view(500, 2)}
    eng.train()
    eng(x)
    (table,) = eng.hashtables().values()
    for block in table._hashtable_impl.emb_blocks()[0]:
        block.normal_()
    trained = {k: v.detach() for k, v in eng(x).items()}
    eng.eval()
    for k, v in eng(x).items():
        torch.testing.assert_close(v, trained[k], rtol=1e-5, atol=1e-5)  # sums of up to 8 rows of N(0, 1) in another order
    with pytest.raises(RuntimeError):
        eng({"b": RaggedTensor(ids(n), off, dense_shape=(499, -1))})


def test_lookup_pool_flags_bad_offsets(rng):
    ht, _ = _table(8, torch.float32, np.arange(10), 64, rng)
    ids = torch.arange(10, device="cuda")
    out = ht._hashtable_impl.lookup_pool_readonly([ids], [torch.tensor([0, 4, 3, 99], device="cuda")], [None], None, False)
    assert out[0].shape == (3, 8) and not out[0].any()
    assert _lib.poll_device_errors() & _lib.DEVERR_OFFSETS


def _offsets(lens):
    return torch.from_numpy(np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)).cuda()


@pytest.mark.parametrize("where", ["this", "earlier", "engine"])
def test_evaluation_raises_what_kernels_reported(where):
    """Evaluation reads no count that error bits could come with: a later call raises them, without a poll by hand."""
    HashtableRegister().clear()
    eng = EmbeddingEngine({"a": EmbeddingOption(embedding_dim=8, block_size=64, shared_name="served", combiner="sum")})
    eng.eval()
    (table,) = eng.hashtables().values()
    table.eval()
    ids = torch.arange(10, device="cuda")
    good = RaggedTensor(ids, _offsets([5, 5]))
    eng({"a": good})
    if where == "this":
        eng({"a": RaggedTensor(ids, torch.tensor([0, 4, 3, 10], device="cuda", dtype=torch.int32))})
    elif where == "earlier":  # another kernel of the device
        ops.segment_reduce_forward(torch.ones(10, 8, device="cuda"), None, None,
                                   torch.tensor([0, 4, 3, 10], device="cuda", dtype=torch.int32), "sum")
        eng({"a": good})
    else:
        for _ in range(3):
            table(ids)
        eng({"a": RaggedTensor(ids, torch.tensor([0, 4, 30, 10], device="cuda", dtype=torch.int32))})
    torch.cuda.synchronize()
    with pytest.raises(RuntimeError, match="offsets not monotone"):
        table(ids) if where == "engine" else eng({"a": good})
    eng({"a": good})
    torch.cuda.synchronize()
    eng({"a": good})
    assert _lib.poll_device_errors() == 0


def test_training_raises_what_evaluation_reported():
    HashtableRegister().clear()
    ht = HashTable([8], block_size=64, name="served")
    ids = torch.arange(10, device="cuda")
    ht(ids)
    ht.eval()
    ops.segment_reduce_forward(torch.ones(10, 8, device="cuda"), None, None,
                               torch.tensor([0, 4, 3, 10], device="cuda", dtype=torch.int32), "sum")
    ht(ids)
    ht.train()
    with pytest.raises(RuntimeError, match="offsets not monotone"):
        ht(ids).sum().backward()
    assert _lib.poll_device_errors() == 0


@pytest.mark.parametrize("D,dtype", [(8192, torch.float32), (8196, torch.float32), (9000, torch.bfloat16)])
def test_evaluation_of_wide_rows(rng, D, dtype):
    ids = torch.arange(6, device="cuda")
    rows = torch.from_numpy(rng.standard_normal((6, D)).astype(np.float32)).cuda().to(dtype)
    tol = dict(rtol=2.0 ** -7 if dtype == torch.bfloat16 else 1e-6, atol=1e-6)
    HashtableRegister().clear()
    table = HashTable([D], block_size=8, dtype=dtype, name="wide")
    table.insert(ids, rows)
    table.eval()
    at = torch.tensor([[3, 1], [5, 77]], device="cuda")
    got = table(at)
    assert torch.equal(got[0, 0], rows[3]) and torch.equal(got[1, 0], rows[5]) and not got[1, 1].any()
    HashtableRegister().clear()
    for module in (DynamicEmbedding(EmbeddingOption(embedding_dim=D, block_size=8, dtype=dtype, shared_name="wide_e")),
                   EmbeddingEngine({"a": EmbeddingOption(embedding_dim=D, block_size=8, dtype=dtype, shared_name="wide_g",
                                                         combiner="mean")})):
        (impl,) = filter_out_sparse_param(module).values()
        impl.insert(ids, rows)
        module.eval()
        x = RaggedTensor(torch.arange(6, device="cuda"), _offsets([2, 0, 4]))
        got = module({"a": x})["a"] if isinstance(module, EmbeddingEngine) else module(x)
        parts = [rows[:2].float().sum(0), torch.zeros(D, device="cuda"), rows[2:].float().sum(0)]
        if isinstance(module, EmbeddingEngine):
            parts = [parts[0] / 2, parts[1], parts[2] / 4]
        torch.testing.assert_close(got, torch.stack(parts).to(dtype), **tol)
    assert _lib.poll_device_errors() == 0


class _Ids(torch.Tensor):
    pass


@pytest.mark.parametrize("training", [False, True])
def test_dense_ids_of_every_kind(rng, training):
    HashtableRegister().clear()
    opt = dict(embedding_dim=8, block_size=64, combiner="sum")
    one = DynamicEmbedding(EmbeddingOption(shared_name="one", **opt)).train(training)
    out = one(torch.empty(7, 0, dtype=torch.int64, device="cuda"))  # no id in any segment
    assert out.shape == (7, 8) and not out.detach().any()
    eng = EmbeddingEngine({"a": EmbeddingOption(shared_name="a", **opt), "b": EmbeddingOption(shared_name="b", **opt)}).train(training)
    (table,) = eng.hashtables().values()
    plain = torch.from_numpy(rng.integers(0, 9, (6, 2))).cuda()
    eng({"a": plain, "b": plain[:, :1]})
    for block in table._hashtable_impl.emb_blocks()[0]:
        block.normal_()
    want = eng({"a": plain, "b": plain[:, :1]})
    for kind in (lambda t: t.as_subclass(_Ids), lambda t: torch.nn.Parameter(t, requires_grad=False), lambda t: t.int(),
                 lambda t: t.cpu()):
        got = eng({"a": kind(plain), "b": kind(plain[:, :1])})
        assert all(torch.equal(got[k], want[k]) for k in want)
    with pytest.raises(Exception):
        eng({"a": torch.empty(7, 0, dtype=torch.int64, device="cuda"), "b": plain[:, :1]})
    with pytest.raises(Exception):
        eng({"a": torch.tensor(3, device="cuda"), "b": plain[:, :1]})
    assert _lib.poll_device_errors() == 0


def test_ids_of_other_types_are_refused_where_they_were():
    """In evaluation HashTable and DynamicEmbedding take int64 ids and do not convert others (a float id has no key)."""
    HashtableRegister().clear()
    table = HashTable([8], block_size=64, name="typed")
    table(torch.arange(4, device="cuda"))
    table.eval()
    one = DynamicEmbedding(EmbeddingOption(embedding_dim=8, block_size=64, shared_name="typed_e"))
    for kind in (torch.int32, torch.float32):
        with pytest.raises((TypeError, RuntimeError)):
            table(torch.arange(4, device="cuda").to(kind))
        with pytest.raises((TypeError, RuntimeError)):
            one.eval()(torch.arange(4, device="cuda").to(kind).view(2, 2))


@pytest.mark.parametrize("lens", [[3, 700, 0, 200, 20], [900, 2500, 1100, 0, 5], [0, 1, 0, 40, 2] * 20])
@pytest.mark.parametrize("weighted", [False, True])
def test_the_last_ids_of_a_feature_of_two_thousand_million(lens, weighted):
    """Ids are numbered up to 2^31 - 2: offsets that name the last ones of such a list."""
    n = 2**31 - 2
    if torch.cuda.mem_get_info()[0] < 16 * n:
        pytest.skip("needs %d GB of device memory" % (16 * n >> 30))
    keys = torch.arange(1, 5000, device="cuda")
    HashtableRegister().clear()
    ht = HashTable([4], block_size=512, name="pool_table")
    rows = torch.randint(-8, 9, (keys.numel(), 4), device="cuda").float()
    ht.insert(keys, rows)
    tail = sum(lens)
    ids = torch.empty(n, dtype=torch.int64, device="cuda")  # only the last ones are ever read
    ids[-tail:] = keys[torch.randint(0, keys.numel(), (tail,), device="cuda")]
    weight = None
    if weighted:
        weight = torch.empty(n, device="cuda")
        weight[-tail:] = torch.randint(-3, 4, (tail,), device="cuda").float()
    off = torch.tensor([n - tail] + lens).cumsum(0).int().cuda()
    got = ht._hashtable_impl.lookup_pool_readonly([ids], [off], [weight], None, False)[0].cpu()
    terms = rows[ids[-tail:] - 1] * (weight[-tail:, None] if weighted else 1)
    want = torch.stack([t.sum(0) if len(t) else torch.zeros(4) for t in torch.split(terms.cpu(), lens)])
    assert torch.equal(got, want)
    assert _lib.poll_device_errors() == 0
