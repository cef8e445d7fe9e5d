"""The training lookups whose forward does not wait for the device (HashtableImpl.lookup_train / dense_lookup_train): counts of
several plans under way at once, errors that come with them, both backward passes over one node."""
import ctypes
import threading

import numpy as np
import pytest
import torch

from recis_amd import _lib, ops
from recis_amd.nn import EmbeddingEngine, EmbeddingOption, HashTable
from recis_amd.nn.hashtable_hook import AdmitHook, FilterHook
from recis_amd.nn.modules.hashtable import HashTableLookupHelpFunction, HashtableRegister, filter_out_sparse_param
from recis_amd.nn.modules.hashtable_hook_impl import HashtableHookFactory
from recis_amd.optim import SparseAdagrad, SparseAdam
from recis_amd.ragged import RaggedTensor

pytestmark = pytest.mark.gpu


def _offsets(lens):
    return torch.from_numpy(np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)).cuda()


@pytest.mark.parametrize("count", [2, 16, 17, 40])
def test_counts_of_plans_under_way_together(rng, count):
    """Every plan's count has a place of its own until it is read, whatever the order."""
    batches = [rng.integers(0, 50 + 37 * k, size=3000) for k in range(count)]
    plans = [ops.ids_unique_plan(torch.from_numpy(b).cuda(), wait=False) for b in batches]
    for k in rng.permutation(count):
        assert plans[k].U == len(np.unique(batches[k]))
    assert _lib.poll_device_errors() == 0


def _trained_table():
    HashtableRegister().clear()
    ht = HashTable([8], block_size=64, name="late")
    return ht, SparseAdagrad(filter_out_sparse_param(ht), lr=0.1)


def test_device_errors_arrive_within_two_steps():
    ht, opt = _trained_table()
    good = torch.arange(100, device="cuda")
    bad = good.clone()
    bad[7] = -1  # a key the map reserves
    with pytest.raises(RuntimeError, match="index outside"):
        for ids in (bad, good, good):
            ht(ids).backward(torch.ones(100, 8, device="cuda"))
            opt.step()
            opt.zero_grad()
    ht(good)
    assert _lib.poll_device_errors() == 0  # raised once, cleared


def test_second_backward_and_no_grad():
    ht, opt = _trained_table()
    ids = torch.arange(50, device="cuda")
    out = ht(ids)
    out.sum().backward(retain_graph=True)
    out.sum().backward()
    with pytest.raises(RuntimeError, match="second time"):
        out.sum().backward()
    opt.step()
    rows = ht._hashtable_impl.lookup_pool_readonly([ids], [None], [None], None, False)[0]
    torch.testing.assert_close(rows, torch.full((50, 8), -0.1, device="cuda"))  # one Adagrad step of a gradient of 2
    with torch.no_grad():
        assert not ht(ids).requires_grad


@pytest.mark.parametrize("weighted", [False, True])
def test_group_of_dense_and_ragged_features_matches_torch(rng, weighted):
    """One group of a dense column, a wide dense tensor and a ragged feature: pooled rows and one Adagrad step against
    index_add_ in float64."""
    HashtableRegister().clear()
    names, D, B = ["a", "b", "c"], 8, 77
    eng = EmbeddingEngine({n: EmbeddingOption(embedding_dim=D, shared_name="one", combiner="sum", use_weight=True)
                           for n in names})
    opt = SparseAdagrad(filter_out_sparse_param(eng), lr=0.1)
    lens = rng.integers(0, 6, size=B)
    off = np.concatenate([[0], np.cumsum(lens)])
    n = int(off[-1])
    ids = {"a": rng.integers(0, 40, size=(B, 1)), "b": rng.integers(0, 40, size=(B, 3)), "c": rng.integers(0, 40, size=n)}
    w = (rng.random(n) + 0.5).astype(np.float32) if weighted else np.ones(n, np.float32)
    x = {k: torch.from_numpy(v).cuda() for k, v in ids.items() if k != "c"}
    x["c"] = RaggedTensor(torch.from_numpy(ids["c"]).cuda(), torch.from_numpy(off.astype(np.int32)).cuda(),
                          torch.from_numpy(w).cuda() if weighted else None)
    (table,) = eng.hashtables().values()
    start = rng.standard_normal((40, D)).astype(np.float32)
    table.insert(torch.arange(40, device="cuda"), torch.from_numpy(start).cuda())
    ups = {k: rng.standard_normal((B, D)).astype(np.float32) for k in names}
    out = eng(x)
    seg = {"a": np.arange(B), "b": np.repeat(np.arange(B), 3), "c": np.repeat(np.arange(B), lens)}
    coef = {"a": np.ones(B), "b": np.ones(3 * B), "c": w.astype(np.float64)}
    grad = np.zeros((40, D))
    for k in names:
        exp = np.zeros((B, D))
        np.add.at(exp, seg[k], coef[k][:, None] * start[ids[k].reshape(-1)].astype(np.float64))
        np.testing.assert_allclose(out[k].detach().cpu().numpy(), exp, rtol=1e-5, atol=1e-5)
        np.add.at(grad, ids[k].reshape(-1), coef[k][:, None] * ups[k][seg[k]])
    torch.autograd.backward([out[k] for k in names], [torch.from_numpy(ups[k]).cuda() for k in names])
    opt.step()
    rows = table._hashtable_impl.lookup_pool_readonly([torch.arange(40, device="cuda")], [None], [None], None, False)[0]
    # the first step moves by lr * sign(g): g is far from zero against its float32 sum
    clear = np.abs(grad) > 1e-3
    np.testing.assert_allclose(rows.cpu().numpy()[clear], (start - 0.1 * np.sign(grad))[clear], rtol=1e-4, atol=1e-4)
    assert _lib.poll_device_errors() == 0


@pytest.mark.parametrize("second", ["tile", "sum"])
def test_step_filter_stamps_rows_of_a_plan_made_without_the_map(rng, second):
    """One input under "mean" with few ids per segment (the general path, whose plan knows no map) and under a combiner
    that takes that plan over: the rows looked up by it are stamped, the gradients of both reach them."""
    HashtableRegister().clear()
    HashtableHookFactory().clear_filters()
    D, B, seq = 8, 60, 4
    common = dict(embedding_dim=D, block_size=64, shared_name="stamped", use_weight=False,
                  filter_hook=FilterHook("GlobalStepFilter", {"filter_step": 5}))
    kw = {"combiner_kwargs": {"tile_len": seq}} if second == "tile" else {}
    eng = EmbeddingEngine({"m": EmbeddingOption(combiner="mean", **common),
                           "x": EmbeddingOption(combiner=second, **kw, **common)})
    eng.train()
    opt = SparseAdagrad(filter_out_sparse_param(eng), lr=0.1)
    (table,) = eng.hashtables().values()
    impl = table._hashtable_impl
    (step_filter,) = [f for fs in HashtableHookFactory().get_filters().values() for f in fs.values()]
    start = rng.standard_normal((30, D)).astype(np.float32)
    impl.insert(torch.arange(30, device="cuda"), torch.from_numpy(start).cuda())
    step_filter.update_step(7)
    lens = rng.integers(1, 4, B)
    ids = rng.integers(0, 25, lens.sum())
    rt = RaggedTensor(torch.from_numpy(ids).cuda(), _offsets(lens))
    out = eng({"m": rt, "x": rt})
    seg = np.repeat(np.arange(B), lens)
    place = np.arange(len(ids)) - np.repeat(np.cumsum(lens) - lens, lens)
    rows = start[ids].astype(np.float64)
    mean = np.zeros((B, D))
    np.add.at(mean, seg, rows / lens[seg][:, None])
    np.testing.assert_allclose(out["m"].detach().cpu().numpy(), mean, rtol=1e-5, atol=1e-6)
    up_m = rng.random((B, D)) + 0.5
    grad = np.zeros((30, D))
    np.add.at(grad, ids, up_m[seg] / lens[seg][:, None])
    if second == "tile":
        up_x = rng.random((B, seq, D)) + 0.5
        padded = np.zeros((B, seq, D))
        padded[seg[place < seq], place[place < seq]] = rows[place < seq]
        np.testing.assert_allclose(out["x"].detach().cpu().numpy().reshape(B, seq, D), padded, rtol=1e-6)
        np.add.at(grad, ids[place < seq], up_x[seg[place < seq], place[place < seq]])
    else:
        up_x = rng.random((B, D)) + 0.5
        total = np.zeros((B, D))
        np.add.at(total, seg, rows)
        np.testing.assert_allclose(out["x"].detach().cpu().numpy(), total, rtol=1e-5, atol=1e-5)
        np.add.at(grad, ids, up_x[seg])
    torch.autograd.backward([out["m"], out["x"]], [torch.from_numpy(up_m.astype(np.float32)).cuda(),
                                                   torch.from_numpy(up_x.astype(np.float32).reshape(B, -1)).cuda()])
    opt.step()
    keys, where = impl.ids_map()
    stamp = torch.cat(impl.get_slot(step_filter._name).kernel_blocks()[0]).view(-1)[where].cpu().numpy()
    accum = torch.cat(impl.get_slot("sparse_adagrad_accum").kernel_blocks()[0])[where].double().cpu().numpy()
    used = np.isin(keys.cpu().numpy(), ids)
    assert (stamp == np.where(used, 7, 0)).all()
    # sums of up to about 20 terms in float32, squared
    np.testing.assert_allclose(accum, grad[keys.cpu().numpy()] ** 2, rtol=2e-5, atol=1e-10)
    HashtableHookFactory().clear_filters()


@pytest.mark.parametrize("kind", ["table", "pool", "tile"])
def test_a_faulty_batch_does_not_reach_the_table(rng, kind):
    """A plan whose kernels report an error (a key the map reserves): its gradient is refused in the backward, before any
    row or any optimizer state is touched."""
    HashtableRegister().clear()
    good = torch.arange(120, device="cuda")
    bad = good.clone()
    bad[7] = -1
    if kind == "table":
        module = HashTable([8], block_size=64, name="late")
        call = lambda ids: module(ids)
    else:
        kw = {"combiner_kwargs": {"tile_len": 5}} if kind == "tile" else {}
        module = EmbeddingEngine({"a": EmbeddingOption(embedding_dim=8, block_size=64, shared_name="late", use_weight=False,
                                                       combiner="sum" if kind == "pool" else "tile", **kw)})
        off = _offsets(np.full(30, 4))
        call = lambda ids: module({"a": RaggedTensor(ids, off)})["a"]
    tables = filter_out_sparse_param(module)
    opt = SparseAdam(tables, lr=0.1)
    (impl,) = tables.values()

    def step(ids):
        out = call(ids)
        out.backward(torch.ones_like(out))
        opt.step()
        opt.zero_grad()

    def state():
        return {s.name(): torch.cat(s.kernel_blocks()[0])[:121].clone() for s in impl.slot_group().slots()}

    step(good)
    before = state()
    with pytest.raises(RuntimeError, match="index outside"):
        step(bad)
    opt.step()
    after = state()
    assert all(torch.equal(before[k], after[k]) for k in before)
    step(good)
    assert _lib.poll_device_errors() == 0
    assert not torch.equal(state()["embedding"], before["embedding"])


@pytest.mark.parametrize("combiner,weighted,what", [("tile", False, "offsets"), ("sum", False, "offsets"), ("sum", True, "weight"),
                                                    ("mean", True, "offsets")])
def test_inputs_refilled_before_the_backward_are_refused(rng, combiner, weighted, what):
    HashtableRegister().clear()
    kw = {"combiner_kwargs": {"tile_len": 5}} if combiner == "tile" else {}
    eng = EmbeddingEngine({"a": EmbeddingOption(embedding_dim=8, block_size=64, shared_name="refilled", use_weight=weighted,
                                                combiner=combiner, **kw)})
    eng.train()
    lens = rng.integers(8, 12, 40)
    off = _offsets(lens)
    n = int(off[-1])
    weight = torch.rand(n, device="cuda") + 0.5 if weighted else None
    out = eng({"a": RaggedTensor(torch.from_numpy(rng.integers(0, 50, n)).cuda(), off, weight)})["a"]
    if what == "weight":
        weight.mul_(2)
    else:
        off.copy_(_offsets(rng.permutation(lens)))
    with pytest.raises(RuntimeError, match="modified by an inplace operation"):
        out.sum().backward()


@pytest.mark.parametrize("combiner", ["tile", "sum", "mean"])
def test_saved_tensor_hooks_see_the_inputs(rng, combiner):
    """What the backward needs of the caller's tensors goes through saved-tensor hooks (offloading, checkpointing)."""
    lens = rng.integers(8, 12, 40)
    ids = rng.integers(0, 50, lens.sum())
    weight = (rng.random(len(ids)) + 0.5).astype(np.float32)
    up = rng.random((40, 8 * (5 if combiner == "tile" else 1))).astype(np.float32)
    got = []
    for hooked in (False, True):
        HashtableRegister().clear()
        kw = {"combiner_kwargs": {"tile_len": 5}} if combiner == "tile" else {}
        eng = EmbeddingEngine({"a": EmbeddingOption(embedding_dim=8, block_size=64, shared_name="offloaded",
                                                    use_weight=combiner != "tile", combiner=combiner, **kw)})
        eng.train()
        opt = SparseAdagrad(filter_out_sparse_param(eng), lr=0.1)
        x = {"a": RaggedTensor(torch.from_numpy(ids).cuda(), _offsets(lens), torch.from_numpy(weight).cuda())}
        packed = []

        def pack(t):
            packed.append((t.dtype, t.numel()))
            return t.cpu()

        if hooked:
            with torch.autograd.graph.saved_tensors_hooks(pack, lambda t: t.cuda()):
                out = eng(x)["a"]
            assert (torch.int32, 41) in packed
            assert combiner == "tile" or (torch.float32, len(ids)) in packed
        else:
            out = eng(x)["a"]
        out.backward(torch.from_numpy(up).cuda())
        opt.step()
        (table,) = eng.hashtables().values()
        table.eval()
        got.append(table(torch.arange(50, device="cuda")))
    assert got[0].any() and torch.equal(got[0], got[1])


def test_errors_of_many_tables_in_one_step(rng):
    """Counts and error bits of more plans than a step of few tables has: each plan's own are there in its backward."""
    HashtableRegister().clear()
    tables = [HashTable([8], block_size=64, name="many%d" % k) for k in range(24)]
    ids = torch.arange(50, device="cuda")
    bad = ids.clone()
    bad[3] = -1

    def step(faulty):
        sum((t(bad if k == faulty else ids)).sum() for k, t in enumerate(tables)).backward()
        for t in tables:
            t.clear_grad()

    step(None)
    with pytest.raises(RuntimeError, match="index outside"):
        step(2)
    step(None)
    assert _lib.poll_device_errors() == 0


def test_a_count_stays_until_it_is_released(rng):
    lib = _lib.lib()
    stream = _lib.stream_ptr()

    def queue(n_distinct, n=3000):
        ids = torch.from_numpy(np.concatenate([np.arange(n_distinct), rng.integers(0, n_distinct, n - n_distinct)])).cuda()
        n = ids.numel()
        cap = n
        out = [torch.empty(n, dtype=torch.int64, device="cuda"), torch.empty(n + 1, dtype=torch.int32, device="cuda"),
               torch.empty(n, dtype=torch.int32, device="cuda"), torch.empty(2 * cap, dtype=torch.int32, device="cuda"),
               torch.empty(2, dtype=torch.int64, device="cuda")]
        p = _lib.ptr
        _lib.check(lib.recis_unique_plan(p(ids), _lib.i64(n), p(out[0]), p(None), p(out[1]), p(out[2]), p(None), p(out[3]),
                                         _lib.i64(cap), p(out[4]), p(None), 1, stream))
        keep.append((ids, out))

    def ticket():
        t = ctypes.c_int64(-1)
        _lib.check(lib.recis_unique_plan_ticket(ctypes.byref(t), stream))
        return t.value

    def count_of(t, wait=1):
        c, bits = ctypes.c_int64(0), ctypes.c_int(0)
        _lib.check(lib.recis_unique_plan_count_of(_lib.i64(t), wait, ctypes.byref(c), ctypes.byref(bits), stream))
        return c.value

    keep = []
    queue(77)
    first = ticket()
    for k in range(60):  # later plans, with a ticket and without one
        queue(100 + k)
        if k % 2:
            t = ticket()
            assert ticket() == -1  # one ticket a count
            assert count_of(t) == 100 + k
            _lib.check(lib.recis_unique_plan_release(_lib.i64(t)))
            assert count_of(t) == -1
    assert count_of(first) == 77
    _lib.check(lib.recis_unique_plan_release(_lib.i64(first)))
    queue(500)
    last = ctypes.c_int64(0)
    _lib.check(lib.recis_unique_plan_count(ctypes.byref(last), stream))
    assert last.value == 500
    # another thread's counts on the stream are its own
    got = []

    def other():
        for k in range(40):
            queue(200 + k)
        t = ticket()
        got.append(count_of(t))
        _lib.check(lib.recis_unique_plan_release(_lib.i64(t)))

    queue(600)
    mine = ticket()
    thread = threading.Thread(target=other)
    thread.start()
    thread.join()
    assert got == [239] and count_of(mine) == 600
    _lib.check(lib.recis_unique_plan_release(_lib.i64(mine)))
    assert _lib.poll_device_errors() == 0


class _TakesNoGradient(torch.autograd.Function):
    @staticmethod
    def forward(ctx, x):
        return x * 1.0

    @staticmethod
    def backward(ctx, g):
        return None


@pytest.mark.parametrize("kind", ["table", "admit", "helper", "engine_dense", "engine_sum", "engine_tile",
                                  "engine_admit"])
def test_no_gradient_for_an_output_counts_as_zeros(rng, kind):
    """A function behind the lookup that returns no gradient for it: the rows of the batch take a gradient of zeros (with
    Adam a step of their momentum), as when autograd hands zeros over."""
    rows = []
    for way in ("none", "zeros"):
        HashtableRegister().clear()
        ids = torch.arange(40, device="cuda")
        if kind.startswith("engine"):
            kw = {"combiner_kwargs": {"tile_len": 5}} if kind == "engine_tile" else {}
            module = EmbeddingEngine({"a": EmbeddingOption(embedding_dim=8, block_size=64, shared_name="nograd", use_weight=False,
                                                           combiner="tile" if kind == "engine_tile" else "sum",
                                                           admit_hook=AdmitHook("ReadOnly") if kind == "engine_admit" else None, **kw)})
            x = ids if kind == "engine_dense" else RaggedTensor(ids, _offsets([4] * 10))
            call = lambda: module({"a": x})["a"]
        else:
            module = HashTable([8], block_size=64, name="nograd", grad_reduce_by="worker")
            admit = AdmitHook("ReadOnly") if kind == "admit" else None
            if kind == "helper":
                call = lambda: HashTableLookupHelpFunction.apply(ids, module._hashtable_impl, module._backward_holder, None)[1]
            else:
                call = lambda: module(ids, admit)
        module.train()
        tables = filter_out_sparse_param(module)
        (impl,) = tables.values()
        impl.insert(ids, torch.ones(40, 8, device="cuda"))
        opt = SparseAdam(tables, lr=0.1)
        out = call()
        out.backward(torch.ones_like(out))
        opt.step()
        opt.zero_grad()
        moved = torch.cat(impl.slot_group().slot_by_name("embedding").kernel_blocks()[0]).clone()
        out = call()
        if way == "none":
            _TakesNoGradient.apply(out).sum().backward()
        else:
            out.backward(torch.zeros_like(out))
        opt.step()
        rows.append(torch.cat(impl.slot_group().slot_by_name("embedding").kernel_blocks()[0]).clone())
        assert not torch.equal(rows[-1], moved)
    assert torch.equal(rows[0], rows[1])


@pytest.mark.parametrize("kinds", ["r", "d", "dd", "rd", "dr", "drdrr", "d" * 50 + "r", "r" * 47 + "dd", "rdz"])
def test_offsets_of_a_group_in_one_launch(rng, kinds):
    """Ragged (r), dense (d) and empty (z) features as one list of offsets."""
    offs, segs, widths, n_ids, want, first = [], [], [], [], [], 0
    for k in kinds:
        s = 0 if k == "z" else int(rng.integers(1, 700))
        if k == "r":
            o = np.concatenate([[0], np.cumsum(rng.integers(0, 5, s))])
            offs.append(torch.from_numpy(o.astype(np.int32)).cuda())
            w = 0
        else:
            w = int(rng.integers(1, 6))
            o = np.arange(s + 1) * w
            offs.append(None)
        want.append(first + o[:-1])
        first += o[-1]
        segs.append(s)
        widths.append(w)
        n_ids.append(int(o[-1]))
    want.append([first])
    want = np.concatenate(want)
    out = torch.full((len(want) + 1,), -7, dtype=torch.int32, device="cuda")
    n = len(kinds)
    arr = lambda v: (ctypes.c_int64 * n)(*v)
    ptrs = (ctypes.c_void_p * n)(*[None if o is None else o.data_ptr() for o in offs])
    call = lambda w: _lib.lib().recis_group_offsets(ptrs, arr(segs), arr(w), arr(n_ids), ctypes.c_int64(n), _lib.ptr(out),
                                                    _lib.stream_ptr())
    assert call(widths) == 0
    assert out[:-1].tolist() == want.tolist() and int(out[-1]) == -7
    if "d" in kinds:
        assert call([w + 1 for w in widths]) != 0  # ids that are not segments of that width


@pytest.mark.parametrize("shape", ["ragged", "mixed"])
def test_as_many_segments_as_ids(rng, shape):
    """As many ids as segments, but not one in each: every gradient goes to the rows of its own segment."""
    HashtableRegister().clear()
    D = 4
    lens = {"a": np.array([0, 2, 1, 0, 3, 0])} if shape == "ragged" else {"a": np.array([0, 3]), "b": np.array([2, 1, 0, 0])}
    assert sum(l.sum() for l in lens.values()) == sum(len(l) for l in lens.values())
    eng = EmbeddingEngine({n: EmbeddingOption(embedding_dim=D, block_size=64, shared_name="s", combiner="sum", use_weight=False)
                           for n in lens})
    eng.train()
    opt = SparseAdagrad(filter_out_sparse_param(eng), lr=0.1)
    (table,) = eng.hashtables().values()
    x, grad, ups, first = {}, np.zeros((6, D)), {}, 0
    for k, l in lens.items():
        ids = np.arange(first, first + l.sum())
        first += l.sum()
        x[k] = RaggedTensor(torch.from_numpy(ids).cuda(), _offsets(l))
        ups[k] = rng.random((len(l), D)).astype(np.float32) + 0.5
        grad[ids] = ups[k][np.repeat(np.arange(len(l)), l)]
    out = eng(x)
    torch.autograd.backward([out[k] for k in x], [torch.from_numpy(ups[k]).cuda() for k in x])
    opt.step()
    keys, where = table._hashtable_impl.ids_map()
    accum = torch.cat(table._hashtable_impl.get_slot("sparse_adagrad_accum").kernel_blocks()[0])[where].cpu().numpy()
    np.testing.assert_allclose(accum, grad[keys.cpu().numpy()] ** 2, rtol=1e-6)


@pytest.mark.parametrize("combiner", ["sum", "tile"])
@pytest.mark.parametrize("kind", ["int64", "int32", "host", "strided", "cube"])
def test_columns_of_one_id_in_every_form(rng, kind, combiner):
    """One id per segment in tensors that the shortest path does not take (other types, places, strides, shapes): rows and
    gradients as for a plain column."""
    HashtableRegister().clear()
    D = 8
    kw = {"combiner_kwargs": {"tile_len": 2}} if combiner == "tile" else {}
    eng = EmbeddingEngine({n: EmbeddingOption(embedding_dim=D, block_size=64, shared_name=n, combiner=combiner, **kw) for n in "ab"})
    eng.train()
    opt = SparseAdagrad(filter_out_sparse_param(eng), lr=0.1)
    ids = rng.integers(0, 9, (20, 1))
    plain = torch.from_numpy(ids).cuda()
    x = {"int64": plain, "int32": plain.int(), "host": plain.cpu(), "strided": torch.cat([plain, plain], 1)[:, :1],
         "cube": plain.view(10, 2, 1)}[kind]
    (table,) = eng.hashtables().values()
    impl = table._hashtable_impl
    keys = torch.cat([torch.arange(9, device="cuda") | (k << 52) for k in range(2)])
    rows = torch.from_numpy(rng.standard_normal((18, D)).astype(np.float32)).cuda()
    impl.insert(keys, rows)
    out = eng({"a": x, "b": x})
    up = torch.rand(20, D, device="cuda") + 0.5
    for k, n in enumerate("ab"):
        got = out[n].reshape(20, -1)
        assert out[n].shape[:-1] == (x.shape[:-1] if kind == "cube" else (20,))
        assert torch.equal(got[:, :D], rows[9 * k + plain.view(-1)]) and not got[:, D:].any()
        got.backward(torch.cat([up, torch.ones_like(got[:, D:])], 1), retain_graph=True)
    opt.step()
    held, where = impl.ids_map()
    accum = torch.cat(impl.get_slot("sparse_adagrad_accum").kernel_blocks()[0])[where][torch.argsort(held)]
    one = torch.zeros(9, D, dtype=torch.float64, device="cuda").index_add_(0, plain.view(-1), up.double())
    torch.testing.assert_close(accum.double(), torch.cat([one, one]) ** 2, rtol=1e-5, atol=0)  # sums of up to 20 terms
    assert _lib.poll_device_errors() == 0


def test_counts_of_threads():
    """Threads that plan batches side by side, each on a stream of its own (calls that share a stream share its scratch memory and
    are queued by one thread at a time): every plan gets its own count."""
    wrong = []

    def work(seed):
        rng = np.random.default_rng(seed)
        with torch.cuda.stream(torch.cuda.Stream()):
            for turn in range(12):
                batches = [rng.integers(0, 20 + int(rng.integers(1, 900)), size=1500) for _ in range(6)]
                plans = [ops.ids_unique_plan(torch.from_numpy(b).cuda(), wait=False) for b in batches]
                for k in rng.permutation(6)[: 6 if turn % 2 else 4]:  # some plans go without being asked
                    if plans[k].U != len(np.unique(batches[k])):
                        wrong.append((seed, turn, int(k)))

    threads = [threading.Thread(target=work, args=(s,)) for s in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not wrong
    assert _lib.poll_device_errors() == 0
