"""What users of this framework have it do, as measurable cases: training steps and read-only lookups through the
embedding modules, the hash table by itself, pooling of materialised rows, and the feature operators.

A case is a dict of plain values whose ``kind`` names one of the workloads below; ``listed()`` gives the fixed ones,
``draw(rng)`` one more of the same ranges. Ids are non-negative 52-bit values (what a coalesced table stores of
them), popularity follows a bounded power law, tables hold more keys than a batch touches and optimizer state is that
of a table part way through training.
"""
import itertools
import math

import numpy as np
import torch

from recis_amd import ops
from recis_amd.features import Bucketize, Feature, FeatureEngine, Hash, IDMultiHash, Mod, SelectField, SequenceTruncate
from recis_amd.nn import EmbeddingEngine, EmbeddingOption, HashTable
from recis_amd.nn.hashtable_hook import FilterHook
from recis_amd.nn.functional.embedding_ops import ragged_embedding_segment_reduce
from recis_amd.nn.modules.hashtable import HashtableRegister, filter_out_sparse_param
from recis_amd.nn.modules.hashtable_hook_impl import HashtableHookFactory
from recis_amd.optim import SparseAdagrad, SparseAdam, SparseAdamW
from recis_amd.ragged import RaggedTensor

DEVICE = "cuda"
_DTYPES = {"float32": torch.float32, "bfloat16": torch.bfloat16, "float16": torch.float16}
_OPTIMIZERS = {"adam": (SparseAdam, 2), "adamw": (SparseAdamW, 2), "adagrad": (SparseAdagrad, 1)}
_serial = itertools.count()


# --------------------------------------------------------------------------------------------- the cases
def listed():
    return [
        # click-through model, one coalesced table of 26 id columns and 13 bucketized float columns, dim 16, Adam:
        # a small batch (online learning: launches and host work count), an ordinary one, the benchmark's batch
        dict(name="ctr_b256", kind="ctr", batch=256, sparse=26, dense=13, dim=16, dtype="float32", optim="adam"),
        dict(name="ctr_b4096", kind="ctr", batch=4096, sparse=26, dense=13, dim=16, dtype="float32", optim="adam"),
        dict(name="ctr_b65536", kind="ctr", batch=65536, sparse=26, dense=13, dim=16, dtype="float32", optim="adam"),
        # one multi-valued id feature, sum pooling, Adagrad (the benchmark's smallest configuration)
        dict(name="ragged_sum_b4096", kind="ragged", features=1, batch=4096, min_len=1, max_len=20, keys=1_000_000,
             alpha=1.05, dim=16, dtype="float32", combiner="sum", weighted=False, optim="adagrad"),
        # several multi-valued features with a weight per value, some of them empty, mean pooling, a row width that is
        # no power of two, AdamW
        dict(name="ragged_weighted_b8192", kind="ragged", features=8, batch=8192, min_len=0, max_len=15, keys=3_000_000,
             alpha=1.05, dim=24, dtype="float32", combiner="mean", weighted=True, optim="adamw"),
        # long behaviour sequences, bfloat16 rows, mean pooled and kept row by row (padded) for an attention
        dict(name="sequence_b2048", kind="sequence", features=4, batch=2048, mean_len=200, max_len=1000,
             keys=50_000_000, alpha=1.2, dim=128, dtype="bfloat16", optim="adagrad"),
        # the hash table by itself at scale: one row per lookup, Adam, last-seen stamps of the step filter
        dict(name="lookup_2m", kind="lookup", ids=2_000_000, resident=20_000_000, alpha=1.1, dim=32, dtype="float32",
             optim="adam"),
        # the same with keys coming and going: a tenth of every batch are keys the table does not hold, every fourth
        # step evicts what was not seen for four steps; the updated rows are read back (evaluation on the batch)
        dict(name="churn_500k", kind="churn", ids=500_000, resident=2_000_000, alpha=1.1, dim=32, dtype="float32",
             optim="adam"),
        # read-only lookups of a trained model: one request, and offline scoring
        dict(name="serve_b256", kind="serve", batch=256, sparse=26, ragged=4, max_len=20, dim=16, dtype="float32"),
        dict(name="serve_b16384", kind="serve", batch=16384, sparse=26, ragged=4, max_len=20, dim=16, dtype="float32"),
        # segment reduce of materialised rows, forward and backward of sum, mean and max (the benchmark's largest)
        dict(name="pool_32x16384", kind="pool", segments=32 * 16384, mean_len=30, dim=64, dtype="float32"),
        # feature operators of an input pipeline: hashed strings, truncated sequences, bucketized floats, multi-hash
        dict(name="features_b8192", kind="features", batch=8192, strings=4, max_strings=20, dense=13, ids=8,
             sequences=4, max_seq=100, multi=2),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["ctr", "ctr", "ragged", "ragged", "sequence", "lookup", "churn", "serve", "serve", "pool",
                       "features"])
    dim = rng.choice([4, 8, 10, 16, 16, 24, 32, 36, 64, 128])
    dtype = rng.choice(["float32", "float32", "bfloat16"])
    if kind == "ctr":
        return dict(kind=kind, batch=_log(rng, 100, 65536), sparse=rng.randint(3, 26), dense=rng.randint(0, 13),
                    dim=min(dim, 32), dtype=dtype, optim=rng.choice(["adam", "adamw", "adagrad"]))
    if kind == "ragged":
        return dict(kind=kind, features=rng.randint(1, 10), batch=_log(rng, 100, 16384), min_len=rng.randint(0, 1),
                    max_len=rng.randint(3, 40), keys=_log(rng, 10_000, 10_000_000), alpha=rng.choice([1.05, 1.1, 1.2]),
                    dim=min(dim, 64), dtype=dtype, combiner=rng.choice(["sum", "mean"]),
                    weighted=rng.choice([False, True]), optim=rng.choice(["adam", "adamw", "adagrad"]))
    if kind == "sequence":
        return dict(kind=kind, features=rng.randint(1, 4), batch=_log(rng, 32, 2048), mean_len=rng.randint(20, 200),
                    max_len=rng.randint(200, 1000), keys=_log(rng, 1_000_000, 50_000_000), alpha=1.2,
                    dim=rng.choice([16, 32, 64, 128]), dtype=dtype if dim < 64 else "bfloat16",
                    optim=rng.choice(["adam", "adagrad"]))
    if kind in ("lookup", "churn"):
        most = 2_000_000 if kind == "lookup" else 500_000
        ids = _log(rng, 5_000, most)
        return dict(kind=kind, ids=ids, resident=_log(rng, 10 * ids, 10 * most) if kind == "lookup" else 4 * ids,
                    alpha=rng.choice([1.05, 1.1, 1.2]), dim=min(dim, 64), dtype=dtype,
                    optim=rng.choice(["adam", "adagrad"]))
    if kind == "serve":
        return dict(kind=kind, batch=_log(rng, 1, 16384), sparse=rng.randint(3, 39), ragged=rng.randint(0, 8),
                    max_len=rng.randint(5, 40), dim=min(dim, 64), dtype=dtype)
    if kind == "pool":
        return dict(kind=kind, segments=_log(rng, 1000, 32 * 16384), mean_len=rng.randint(6, 30),
                    dim=min(dim, 64), dtype=dtype)
    return dict(kind=kind, batch=_log(rng, 100, 16384), strings=rng.randint(2, 5), max_strings=rng.randint(2, 30),
                dense=rng.randint(1, 13), ids=rng.randint(1, 10), sequences=rng.randint(2, 5),
                max_seq=rng.randint(20, 200), multi=rng.randint(1, 2))


# --------------------------------------------------------------------------------------------- inputs
def _mix(x):
    """A bijective mix of int64 values, cut to 52 bits: ranks become keys."""
    x = x * -7046029254386353131
    x = torch.bitwise_xor(x, torch.bitwise_and(x >> 29, (1 << 35) - 1)) * -4658895280553007687
    return torch.bitwise_and(x >> 11, (1 << 52) - 1)


def _power_law(n, keys, alpha, gen):
    """n ranks in [0, keys), popularity of rank r about (r + 1) ** -alpha."""
    u = torch.rand(n, dtype=torch.float64, device=DEVICE, generator=gen)
    e = 1.0 - alpha
    r = ((keys ** e - 1.0) * u + 1.0).pow_(1.0 / e).to(torch.int64).sub_(1)
    return r.clamp_(0, keys - 1)


def _distinct(n, keys, alpha):
    """Expected number of distinct ranks among n draws of ``_power_law``."""
    e = 1.0 - alpha
    edge = np.unique(np.round(np.geomspace(1, keys + 1, 4000))).astype(np.float64)
    width = edge[1:] - edge[:-1]
    p = (edge[1:] ** e - edge[:-1] ** e) / ((keys + 1.0) ** e - 1.0) / width
    return float(np.sum(width * -np.expm1(n * np.log1p(-p))))


def _cardinality(field):
    """Log-uniform over 10 .. 1e7, spread evenly over the fields."""
    return int(10 ** (1 + 6 * ((field * 0.6180339887) % 1.0)))


def _offsets(lens):
    off = torch.zeros(lens.numel() + 1, dtype=torch.int32, device=DEVICE)
    off[1:] = torch.cumsum(lens, 0)
    return off


def _lengths(count, min_len, max_len, gen):
    """Lengths spread evenly over min_len .. max_len, in an order of the seed's: their sum is the case's alone."""
    even = torch.arange(count, device=DEVICE) % (max_len - min_len + 1) + min_len
    return even[torch.randperm(count, device=DEVICE, generator=gen)]


def _ragged(batch, min_len, max_len, keys, alpha, gen, field, weighted=False):
    off = _offsets(_lengths(batch, min_len, max_len, gen))
    n = int(off[-1])
    values = _mix(_power_law(n, keys, alpha, gen) + field * keys)
    weight = torch.rand(n, device=DEVICE, generator=gen) + 0.5 if weighted else None
    return RaggedTensor(values, off, weight)


def _insert(table, keys, dtype, gen):
    """Admits ``keys`` (duplicates removed) with rows N(0, 0.01), a piece at a time as a loader does: a table that was
    given its size makes room for sixteen more calls as large as one that asks for a large part of it."""
    keys = torch.unique(keys)
    piece = max(1, table.slot_group().chunk_rows() // 33)
    for part in torch.split(keys, piece):
        rows = torch.randn([part.numel()] + list(table.embedding_shape()), device=DEVICE, generator=gen).mul_(0.01)
        table.insert(part, rows.to(dtype))


def _train_part_way(table, gen):
    """Optimizer state as after some training: second moments / accumulators away from zero."""
    for slot in table.slot_group().slots()[1:]:
        if not slot.name().startswith("sparse_"):
            continue
        for block in slot.kernel_blocks()[0]:
            block.normal_(0, 0.1, generator=gen)
            if not slot.name().endswith("exp_avg"):
                block.square_().add_(0.05)


def _state_of(table):
    """Every row of every float slot of a table: the parameters and the optimizer's state."""
    out = []
    for slot in table.slot_group().slots():
        blocks = slot.kernel_blocks()[0]
        if blocks[0].is_floating_point():
            out += blocks
    return out


def _engine(options, training):
    HashtableRegister().clear()
    engine = EmbeddingEngine(options)
    engine.train(training)
    return engine


def _table_of(engine):
    (table,) = engine.hashtables().values()
    return table


def _optimizer(case, module, gen):
    tables = filter_out_sparse_param(module)
    opt = _OPTIMIZERS[case["optim"]][0](tables, lr=1e-3)
    for table in tables.values():
        _train_part_way(table, gen)
    return opt


def _boundaries(count=64):
    q = torch.linspace(0.5 / count, 1 - 0.5 / count, count, dtype=torch.float64)
    return torch.exp(2.0 * math.sqrt(2.0) * torch.erfinv(2 * q - 1)).float()


def _encoded(engine, names, columns):
    """The keys a coalesced table stores for the ids of its features."""
    info = _table_of(engine)._hashtable_impl.children_info()
    if not info.is_coalesce():
        return torch.cat(columns)
    return ops.ids_encode(columns, [info.child_index(n) for n in names])


def prepare(case, seed):
    gen = torch.Generator(device=DEVICE).manual_seed(seed)
    torch.manual_seed(seed)
    state = _PREPARE[case["kind"]](case, gen)
    state["case"] = case
    return state


def run(state):
    return _RUN[state["case"]["kind"]](state)


# --------------------------------------------------------------------------------------------- ctr
def _prepare_ctr(case, gen):
    batch, dim, dtype = case["batch"], case["dim"], _DTYPES[case["dtype"]]
    sparse = ["s%d" % i for i in range(case["sparse"])]
    dense = ["d%d" % i for i in range(case["dense"])]
    names = sparse + dense
    cards = [_cardinality(i) for i in range(len(sparse))]

    def columns():
        return [torch.randint(0, c, (batch, 1), device=DEVICE, generator=gen) for c in cards]

    bounds = _boundaries().to(DEVICE)
    features = FeatureEngine([Feature(n).add_op(SelectField(n)).add_op(Bucketize(bounds)).add_op(Mod(1_000_000))
                              for n in dense]) if dense else None
    floats = {n: torch.randn(batch, device=DEVICE, generator=gen).mul_(2).exp_() for n in dense}
    inputs = dict(zip(sparse, columns()))
    # the table holds the keys of four batches and every bucket
    held = [inputs] + [dict(zip(sparse, columns())) for _ in range(3)]
    buckets = torch.arange(len(bounds) + 1, device=DEVICE)
    engine = _engine({n: EmbeddingOption(embedding_dim=dim, dtype=dtype, shared_name=n, combiner="sum", use_weight=False,
                                         reserve_rows=12 * batch + 128) for n in names}, True)
    keys = torch.cat([_encoded(engine, names, [h[n].view(-1) for n in sparse] + [buckets] * len(dense)) for h in held])
    table = _table_of(engine)._hashtable_impl
    _insert(table, keys, dtype, gen)
    opt = _optimizer(case, engine, gen)
    up = torch.randn((batch, dim * len(names)), device=DEVICE, generator=gen).mul_(0.1).to(dtype)
    return dict(engine=engine, features=features, inputs=inputs, floats=floats, names=names, opt=opt, up=up, table=table)




def _train_step(s, data):
    """Lookup and pooling, the outputs side by side as a dense tower takes them, backward, optimizer step."""
    out = s["engine"](data)
    tower = torch.cat([out[n] for n in s["names"]], dim=1)
    tower.backward(s["up"])
    s["opt"].step()
    s["opt"].zero_grad()
    return [tower.detach()] + _state_of(s["table"])


def _run_ctr(s):
    data = dict(s["inputs"])
    if s["features"] is not None:
        data.update(s["features"](s["floats"]))
    return _train_step(s, data)


# --------------------------------------------------------------------------------------------- ragged
def _prepare_ragged(case, gen):
    dtype, dim, batch = _DTYPES[case["dtype"]], case["dim"], case["batch"]
    names = ["f%d" % i for i in range(case["features"])]

    def draw_batch():
        return {n: _ragged(batch, case["min_len"], case["max_len"], case["keys"], case["alpha"], gen, i,
                           case["weighted"]) for i, n in enumerate(names)}

    inputs = draw_batch()
    held = [inputs] + [draw_batch() for _ in range(3)]
    engine = _engine({n: EmbeddingOption(embedding_dim=dim, dtype=dtype, shared_name=n, combiner=case["combiner"],
                                         use_weight=case["weighted"], reserve_rows=6 * batch * (case["max_len"] + 2))
                      for n in names}, True)
    table = _table_of(engine)._hashtable_impl
    _insert(table, torch.cat([_encoded(engine, names, [h[n].values() for n in names]) for h in held]), dtype, gen)
    opt = _optimizer(case, engine, gen)
    up = torch.randn((batch, dim * len(names)), device=DEVICE, generator=gen).mul_(0.1).to(dtype)
    return dict(engine=engine, inputs=inputs, names=names, opt=opt, up=up, table=table)


def _run_ragged(s):
    return _train_step(s, s["inputs"])


# --------------------------------------------------------------------------------------------- sequence
def _prepare_sequence(case, gen):
    dtype, dim, batch, longest = _DTYPES[case["dtype"]], case["dim"], case["batch"], case["max_len"]
    options, inputs, names = {}, {}, []
    reserve = 10 * batch * case["mean_len"]
    for i in range(case["features"]):
        lens = torch.randn(batch, device=DEVICE, generator=gen).add_(math.log(case["mean_len"]) - 0.5).exp_()
        off = _offsets(lens.round_().clamp_(1, longest).to(torch.int64))
        values = _mix(_power_law(int(off[-1]), case["keys"], case["alpha"], gen) + i * case["keys"])
        common = dict(embedding_dim=dim, dtype=dtype, shared_name="q%d" % i, use_weight=False, reserve_rows=reserve // 2)
        options["mean%d" % i] = EmbeddingOption(combiner="mean", **common)
        options["rows%d" % i] = EmbeddingOption(combiner="tile", combiner_kwargs={"tile_len": longest}, **common)
        inputs["mean%d" % i] = inputs["rows%d" % i] = RaggedTensor(values, off)
        names.append("q%d" % i)
    engine = _engine(options, True)
    table = _table_of(engine)._hashtable_impl
    _insert(table, _encoded(engine, names, [inputs["mean%d" % i].values() for i in range(len(names))]), dtype, gen)
    opt = _optimizer(case, engine, gen)
    ups = {}
    for i in range(len(names)):
        ups["mean%d" % i] = torch.randn((batch, dim), device=DEVICE, generator=gen).to(dtype)
        ups["rows%d" % i] = torch.randn((batch, longest * dim), device=DEVICE, dtype=torch.bfloat16 if
                                        dtype == torch.bfloat16 else torch.float32, generator=gen).mul_(0.1).to(dtype)
    return dict(engine=engine, inputs=inputs, opt=opt, ups=ups, table=table)


def _run_sequence(s):
    out = s["engine"](s["inputs"])
    order = sorted(out)
    torch.autograd.backward([out[k] for k in order], [s["ups"][k] for k in order])
    s["opt"].step()
    s["opt"].zero_grad()
    return [out[k].detach() for k in order] + _state_of(s["table"])


# --------------------------------------------------------------------------------------------- lookup, churn
def _hash_table(case, reserve, filter_step):
    HashtableRegister().clear()
    name = "table%d" % next(_serial)
    table = HashTable([case["dim"]], block_size=10240, dtype=_DTYPES[case["dtype"]], name=name, children=[name],
                      filter_hook=FilterHook("GlobalStepFilter", {"filter_step": filter_step}), reserve_rows=reserve)
    table.train()
    factory = HashtableHookFactory()
    (step_filter,) = factory.get_filters()[name].values()
    factory.clear_filters()
    return table, step_filter


def _prepare_lookup(case, gen):
    n, resident = case["ids"], case["resident"]
    table, step_filter = _hash_table(case, resident + 8 * n, 1000)
    _insert(table._hashtable_impl, _mix(torch.arange(resident, device=DEVICE)), _DTYPES[case["dtype"]], gen)
    opt = _optimizer(case, table, gen)
    ids = _mix(_power_law(n, resident, case["alpha"], gen))
    up = torch.randn((n, case["dim"]), device=DEVICE, generator=gen).mul_(0.1).to(_DTYPES[case["dtype"]])
    return dict(table=table, step_filter=step_filter, ids=ids, up=up, opt=opt)


def _run_lookup(s):
    out = s["table"](s["ids"])
    out.backward(s["up"])
    s["opt"].step()
    s["opt"].zero_grad()
    s["step_filter"].update_step()
    return [out.detach()] + _state_of(s["table"]._hashtable_impl)


_CHURN_BATCHES, _CHURN_EVERY = 8, 4


def _prepare_churn(case, gen):
    n, resident = case["ids"], case["resident"]
    table, step_filter = _hash_table(case, resident + 2 * _CHURN_BATCHES * n, _CHURN_EVERY)
    _insert(table._hashtable_impl, _mix(torch.arange(resident, device=DEVICE)), _DTYPES[case["dtype"]], gen)
    opt = _optimizer(case, table, gen)
    batches = []
    for k in range(_CHURN_BATCHES):
        ranks = _power_law(n, resident, case["alpha"], gen)
        fresh = n // 10
        at = torch.randperm(n, device=DEVICE, generator=gen)[:fresh]
        ranks[at] = resident + k * fresh + torch.arange(fresh, device=DEVICE)
        batches.append(_mix(ranks))
    # rows that leave are handed out again as their initialiser made them: state of zero, rows of zero
    for slot in table.slot_group().slots():
        if slot.name().startswith("sparse_"):
            for block in slot.kernel_blocks()[0]:
                block.zero_()
    up = torch.rand((n, case["dim"]), device=DEVICE, generator=gen).add_(0.5).to(_DTYPES[case["dtype"]])
    return dict(table=table, step_filter=step_filter, batches=batches, up=up, opt=opt, turn=0)


def _run_churn(s):
    table, ids = s["table"], s["batches"][s["turn"] % _CHURN_BATCHES]
    s["turn"] += 1
    out = table(ids)
    out.backward(s["up"])
    s["opt"].step()
    s["opt"].zero_grad()
    s["step_filter"].update_step()
    if s["turn"] % _CHURN_EVERY == 0:
        s["step_filter"].do_filter()
    table.eval()
    after = table(ids)
    table.train()
    return [out.detach(), after]


# --------------------------------------------------------------------------------------------- serve
def _prepare_serve(case, gen):
    batch, dtype, dim = case["batch"], _DTYPES[case["dtype"]], case["dim"]
    sparse = ["s%d" % i for i in range(case["sparse"])]
    ragged = ["r%d" % i for i in range(case["ragged"])]
    names = sparse + ragged
    cards = [_cardinality(i) for i in range(len(sparse))]
    inputs = {n: torch.randint(0, c, (batch, 1), device=DEVICE, generator=gen) for n, c in zip(sparse, cards)}
    for i, n in enumerate(ragged):
        inputs[n] = _ragged(batch, 0, case["max_len"], 1_000_000, 1.05, gen, i)
    engine = _engine({n: EmbeddingOption(embedding_dim=dim, dtype=dtype, shared_name=n, combiner="sum", use_weight=False,
                                         reserve_rows=100_000) for n in names}, False)
    table = _table_of(engine)._hashtable_impl
    # the model has seen every key of the small columns, 100 000 keys of the large ones, and most of this batch
    seen = [torch.randint(0, c, (min(c, 50_000),), device=DEVICE, generator=gen) for c in cards]
    seen = [torch.cat([a, inputs[n].view(-1)[: 9 * batch // 10]]) for a, n in zip(seen, sparse)]
    seen += [inputs[n].values()[: 9 * inputs[n].values().numel() // 10] for n in ragged]
    _insert(table, _encoded(engine, names, seen), dtype, gen)
    return dict(engine=engine, inputs=inputs, names=names)


def _run_serve(s):
    with torch.no_grad():
        out = s["engine"](s["inputs"])
        return torch.cat([out[n] for n in s["names"]], dim=1)


# --------------------------------------------------------------------------------------------- pool
def _prepare_pool(case, gen):
    # every segment holds one value; the others fall into segments at random (Poisson lengths with a sum of the case's)
    more = torch.randint(0, case["segments"], (case["segments"] * (case["mean_len"] - 1),), device=DEVICE, generator=gen)
    off = _offsets(torch.bincount(more, minlength=case["segments"]) + 1)
    dtype = _DTYPES[case["dtype"]]
    values = torch.randn((int(off[-1]), case["dim"]), device=DEVICE, generator=gen).to(dtype).requires_grad_(True)
    grad = torch.randn((case["segments"], case["dim"]), device=DEVICE, generator=gen).to(dtype)
    return dict(values=values, offsets=off, grad=grad)


def _run_pool(s):
    res = []
    for combiner in ("sum", "mean", "max"):
        out = ragged_embedding_segment_reduce(s["values"], None, None, s["offsets"], combiner)
        res += [out.detach(), torch.autograd.grad(out, s["values"], s["grad"].to(out.dtype))[0]]
    return res


# --------------------------------------------------------------------------------------------- features
def _prepare_features(case, gen):
    batch, data, features = case["batch"], {}, []
    for i in range(case["strings"]):
        outer = _offsets(_lengths(batch, 1, case["max_strings"], gen))
        inner = _offsets(_lengths(int(outer[-1]), 4, 24, gen))
        data["h%d" % i] = RaggedTensor(torch.randint(32, 127, (int(inner[-1]),), device=DEVICE, dtype=torch.int8,
                                                     generator=gen), [outer, inner])
        features.append(Feature("h%d" % i).add_op(SelectField("h%d" % i)).add_op(Hash("farm" if i % 2 else "murmur"))
                        .add_op(SequenceTruncate(max(1, case["max_strings"] // 2), check_length=False)))
    for i in range(case["sequences"]):
        data["q%d" % i] = _ragged(batch, 0, case["max_seq"], 10_000_000, 1.1, gen, i)
        features.append(Feature("q%d" % i).add_op(SelectField("q%d" % i)).add_op(Mod(2_000_003 + i))
                        .add_op(SequenceTruncate(max(1, case["max_seq"] // 2), check_length=False,
                                                 truncate_side="left" if i % 2 else "right")))
    bounds = _boundaries().to(DEVICE)
    for i in range(case["dense"]):
        data["d%d" % i] = torch.randn(batch, device=DEVICE, generator=gen).mul_(2).exp_()
        features.append(Feature("d%d" % i).add_op(SelectField("d%d" % i)).add_op(Bucketize(bounds * (1 + i)))
                        .add_op(Mod(1_000_000)))
    for i in range(case["ids"]):
        data["m%d" % i] = _mix(torch.randint(0, 1 << 40, (batch,), device=DEVICE, generator=gen))
        features.append(Feature("m%d" % i).add_op(SelectField("m%d" % i)).add_op(Mod(1_000_003 + i)))
    for i in range(case["multi"]):
        data["x%d" % i] = torch.randint(0, 1 << 40, (batch,), device=DEVICE, generator=gen)
        features.append(Feature("x%d" % i).add_op(SelectField("x%d" % i))
                        .add_op(IDMultiHash([100_003 + i] * 4, prefix="x%d_hash" % i)))
    return dict(engine=FeatureEngine(features), data=data)


def _run_features(s):
    res = []
    for name, value in s["engine"](s["data"], remain_no_use_data=False).items():
        res += [value.values(), value.offsets()[-1]] if isinstance(value, RaggedTensor) else [value]
    return res


_PREPARE = {"ctr": _prepare_ctr, "ragged": _prepare_ragged, "sequence": _prepare_sequence, "lookup": _prepare_lookup,
            "churn": _prepare_churn, "serve": _prepare_serve, "pool": _prepare_pool, "features": _prepare_features}
_RUN = {"ctr": _run_ctr, "ragged": _run_ragged, "sequence": _run_sequence, "lookup": _run_lookup, "churn": _run_churn,
        "serve": _run_serve, "pool": _run_pool, "features": _run_features}


# --------------------------------------------------------------------------------------------- work, tolerance
def _update_bytes(case, distinct, row):
    """Per distinct key of a training step: its slot of the map, its row and optimizer state read and written."""
    return distinct * (16 + 2 * row * (1 + _OPTIMIZERS[case["optim"]][1]))


def work(case):
    kind = case["kind"]
    size = 4 if case.get("dtype", "float32") == "float32" else 2
    row = case.get("dim", 0) * size
    if kind == "ctr":
        n = case["batch"] * (case["sparse"] + case["dense"])
        distinct = sum(c * -math.expm1(-case["batch"] / c) for c in map(_cardinality, range(case["sparse"])))
        distinct += case["dense"] * min(65, case["batch"])
        return {"bytes": 8 * case["batch"] * case["sparse"] + 4 * case["batch"] * case["dense"] + 2 * n * row
                + _update_bytes(case, distinct, row), "flops": 2 * n * case["dim"]}
    if kind == "ragged":
        n = case["features"] * case["batch"] * (case["min_len"] + case["max_len"]) / 2
        distinct = case["features"] * _distinct(n / case["features"], case["keys"], case["alpha"])
        return {"bytes": n * (12 if case["weighted"] else 8) + case["features"] * case["batch"] * (4 + 2 * row)
                + _update_bytes(case, distinct, row), "flops": 4 * n * case["dim"]}
    if kind == "sequence":
        n = case["features"] * case["batch"] * case["mean_len"] * 0.95
        distinct = case["features"] * _distinct(n / case["features"], case["keys"], case["alpha"])
        padded = case["features"] * case["batch"] * case["max_len"]
        # the padded rows are written whole, their gradient is read where there is an id
        return {"bytes": 8 * n + case["features"] * case["batch"] * (4 + 2 * row) + padded * row + n * row
                + _update_bytes(case, distinct, row), "flops": 6 * n * case["dim"]}
    if kind in ("lookup", "churn"):
        n = case["ids"] * (0.9 if kind == "churn" else 1.0)
        distinct = _distinct(n, case["resident"], case["alpha"]) + (case["ids"] - n)
        total = case["ids"] * (8 + 2 * row) + _update_bytes(case, distinct, row) + 8 * distinct
        if kind == "churn":  # the evaluation reads ids and rows again; a quarter of a sweep over the keys held
            total += case["ids"] * (8 + row) + distinct * (16 + row)
        return {"bytes": total, "flops": 2 * case["ids"] * case["dim"]}
    if kind == "serve":
        values = case["batch"] * case["ragged"] * case["max_len"] / 2
        segments = case["batch"] * (case["sparse"] + case["ragged"])
        distinct = sum(c * -math.expm1(-case["batch"] / c) for c in map(_cardinality, range(case["sparse"])))
        distinct += case["ragged"] * _distinct(values / max(1, case["ragged"]), 1_000_000, 1.05)
        return {"bytes": 8 * (case["batch"] * case["sparse"] + values) + 4 * case["ragged"] * case["batch"]
                + distinct * (16 + row) + segments * row, "flops": values * case["dim"]}
    if kind == "pool":
        n = case["segments"] * case["mean_len"]
        one = n * row + case["segments"] * (4 + row)
        return {"bytes": 6 * one + 2 * case["segments"] * case["dim"] * 4, "flops": 6 * n * case["dim"]}
    strings = case["batch"] * case["strings"] * (case["max_strings"] + 1) / 2
    values = case["batch"] * case["sequences"] * case["max_seq"] / 2
    return {"bytes": strings * (14 + 4 + 8 * 0.75) + values * (8 + 8 * 0.75) + 8 * case["batch"] *
            (case["strings"] + case["sequences"]) + case["batch"] * (12 * case["dense"] + 16 * case["ids"] + 40 *
                                                                     case["multi"]), "flops": 20 * (strings + values)}


def tolerance(case):
    """Hashes, buckets and offsets are whole numbers. float32: the steps against themselves with the batch in reverse
    order (every sum in another order) differ by up to 1.5e-7 in norm and 7e-6 in one value, pooling against 64-bit
    sums by 8e-8 and 6e-7; a sum that nearly cancels differs by more. bfloat16: by one rounding of values that lie at the
    edge between two of the type's (8e-3), in norm by 2e-6 to 1e-4."""
    if case["kind"] == "features":
        return "exact"
    if case["dtype"] == "float32":
        return {"rel": 2e-6, "max": 2e-4}
    return {"rel": 1e-3, "max": 3e-2}
