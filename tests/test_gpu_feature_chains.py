"""Feature engines whose chains run in one native call against the same engines operator by operator."""
import pytest
import torch

from recis_amd import _lib
from recis_amd.features import Bucketize, Feature, FeatureEngine, Hash, IDMultiHash, Mod, SelectField, SequenceTruncate
from recis_amd.ragged import RaggedTensor

pytestmark = pytest.mark.gpu


def _offsets(rng, rows, longest, dtype):
    lens = torch.from_numpy(rng.integers(0, longest + 1, size=rows))
    off = torch.zeros(rows + 1, dtype=torch.int64)
    off[1:] = torch.cumsum(lens, 0)
    return off.to(dtype)


def _data(rng, rows, off_dtype):
    outer = _offsets(rng, rows, 5, off_dtype)
    inner = _offsets(rng, int(outer[-1]), 30, off_dtype)
    text = torch.from_numpy(rng.integers(32, 127, size=int(inner[-1]))).to(torch.int8)
    seq = _offsets(rng, rows, 9, off_dtype)
    ids = torch.from_numpy(rng.integers(-(2**62), 2**62, size=int(seq[-1])))
    weight = torch.rand(ids.numel())
    data = {"text": RaggedTensor(text, [outer, inner]), "seq": RaggedTensor(ids, seq, weight),
            "wide": torch.from_numpy(rng.integers(0, 2**40, size=(rows, 3))),
            "strided": torch.from_numpy(rng.integers(0, 2**40, size=(3, rows))).t(), "one": torch.arange(rows)[::2],
            "real": torch.randn(rows, 2), "real_off": torch.randn(2 * rows + 1)[1:], "untouched": torch.arange(3)}
    return {k: v.cuda() for k, v in data.items()}


def _features():
    bounds = torch.linspace(-2, 2, 33)
    sel = lambda name, src: Feature(name).add_op(SelectField(src))
    cut = lambda n, side="right": SequenceTruncate(n, check_length=False, truncate_side=side)
    return [sel("farm", "text").add_op(Hash("farm")), sel("farm_cut", "text").add_op(Hash("farm")).add_op(cut(2)),
            sel("murmur_cut", "text").add_op(Hash("murmur")).add_op(cut(3, "left")),
            sel("seq", "seq").add_op(Mod(1009)), sel("seq_cut", "seq").add_op(Mod(77)).add_op(cut(4, "left")),
            sel("raw_cut", "seq").add_op(cut(1)), sel("nothing_left", "seq").add_op(cut(0)), sel("as_is", "wide"),
            sel("wide", "wide").add_op(Mod(10)), sel("strided", "strided").add_op(Mod(13)), sel("one", "one").add_op(Mod(3)),
            sel("same", "wide").add_op(Mod(10)),
            sel("bucket", "real").add_op(Bucketize(bounds)).add_op(Mod(20)),
            sel("bucket_off", "real_off").add_op(Bucketize(bounds.cuda())).add_op(Mod(1000)),
            sel("multi", "strided").add_op(IDMultiHash([101, 103], prefix="m")),
            sel("multi_seq", "seq").add_op(IDMultiHash([1001] * 4, prefix="ms"))]


def _same(a, b):
    assert type(a) is type(b)
    if isinstance(a, RaggedTensor):
        assert a.dense_shape == b.dense_shape and len(a.offsets()) == len(b.offsets())
        _same(a.values(), b.values())
        for x, y in zip(a.offsets(), b.offsets()):
            _same(x, y)
        assert (a.weight() is None) == (b.weight() is None) and (a.weight() is None or a.weight() is b.weight())
        assert (a.pad_info is None) == (b.pad_info is None)
        if a.pad_info is not None:
            for field in ("drop_nums", "pad_nums", "drop_sides", "pad_sides"):
                _same(getattr(a.pad_info, field), getattr(b.pad_info, field))
    else:
        assert a.dtype == b.dtype and a.device == b.device and a.shape == b.shape and torch.equal(a, b)


def _both(features, data, **kw):
    one_call, by_op = FeatureEngine(features()), FeatureEngine(features())
    assert one_call._chains is not None
    by_op._chains = None
    got, want = one_call(data, **kw), by_op(data, **kw)
    assert list(got) == list(want)
    for name in want:
        _same(got[name], want[name])
    return one_call


@pytest.mark.parametrize("rows", [1, 2, 257, 5000])
@pytest.mark.parametrize("off_dtype", [torch.int32, torch.int64])
def test_chains_equal_the_operators_one_by_one(rng, rows, off_dtype):
    data = _data(rng, rows, off_dtype)
    engine = _both(_features, data)
    assert engine._chains.run(data) is not None
    _both(_features, data, remain_no_use_data=False)
    _both(lambda: [f for f in _features() if f.name in ("wide", "same", "murmur_cut", "bucket", "multi")], data)  # one of a kind
    assert _lib.poll_device_errors() == 0


def test_outputs_do_not_share_a_version(rng):
    out = FeatureEngine(_features())(_data(rng, 50, torch.int64))
    before = out["wide"]._version, out["farm_cut"].values()._version, out["m_1"]._version
    out["strided"].add_(1)
    out["seq_cut"].values().add_(1)
    out["m_0"].add_(1)
    assert (out["wide"]._version, out["farm_cut"].values()._version, out["m_1"]._version) == before


def test_multi_hashes_have_storages_of_their_own(rng):
    out = FeatureEngine(_features())(_data(rng, 50, torch.int64))
    hashes = [out["m_%d" % j] for j in range(2)] + [out["ms_%d" % j].values() for j in range(4)]
    assert all(h.untyped_storage().nbytes() == 8 * h.numel() for h in hashes)
    assert len({h.untyped_storage().data_ptr() for h in hashes}) == 6


def test_what_the_call_does_not_take_runs_operator_by_operator(rng):
    data = _data(rng, 40, torch.int64)
    on_host = {k: (v.cpu() if k in ("wide", "real") else v) for k, v in data.items()}
    assert _both(_features, on_host)._chains.run(on_host) is None
    mixed = dict(data, seq=RaggedTensor(data["seq"].values(), data["seq"].offsets()[0].int()))
    assert FeatureEngine(_features())._chains.run(mixed) is None
    hooked = FeatureEngine(_features())
    calls = []
    hooked._features["wide"].ops[0].register_forward_hook(lambda *a: calls.append(1))
    hooked(data)
    assert calls == [1]
    with pytest.raises(TypeError):
        FeatureEngine(_features())(dict(data, wide=data["wide"].int()))
    with pytest.raises(KeyError):
        FeatureEngine(_features())({k: v for k, v in data.items() if k != "real"})
    checked = lambda: [Feature("s").add_op(SelectField("seq")).add_op(SequenceTruncate(2))]
    with pytest.raises(AssertionError):
        FeatureEngine(checked())(data)
    other = [Feature("b").add_op(SelectField("real")).add_op(Bucketize([0.0]))]
    assert FeatureEngine(other)._chains is None
    plain = FeatureEngine([Feature("as_is").add_op(SelectField("wide"))])  # nothing for the call to do
    assert plain._chains is None and plain(data)["as_is"] is data["wide"]


def test_more_columns_than_a_launch_takes_and_long_boundaries(rng):
    data = {"c%d" % k: torch.from_numpy(rng.integers(-(2**62), 2**62, size=int(n))).cuda()
            for k, n in enumerate(rng.integers(0, 4000, size=60))}
    data.update({"r%d" % k: torch.randn(3001).cuda() for k in range(4)})
    mods = [1, 2, 2**31 - 1, 2**31, 2**32 - 1, 2**32, 2**40 + 3, -5]

    def features():
        out = [Feature("c%d" % k).add_op(SelectField("c%d" % k)).add_op(Mod(mods[k % len(mods)])) for k in range(60)]
        for k, n in enumerate((0, 2048, 2049, 9000)):
            bounds = torch.sort(torch.randn(n, generator=torch.Generator().manual_seed(k))).values
            out.append(Feature("r%d" % k).add_op(SelectField("r%d" % k)).add_op(Bucketize(bounds)).add_op(Mod(700)))
        return out

    _both(features, data)
    assert _lib.poll_device_errors() == 0


@pytest.mark.parametrize("mods", [[2**63 + 5], [2**64 - 59], [2**63, 2**63 - 1, 2**64 - 1, 2**64 + 7, 2**63 + 1]])
def test_moduli_are_any_uint64(rng, mods):
    data = {"c%d" % k: torch.from_numpy(rng.integers(-(2**63), 2**63 - 1, size=300)).cuda() for k in range(len(mods))}
    features = lambda: [Feature("c%d" % k).add_op(SelectField("c%d" % k)).add_op(Mod(m)) for k, m in enumerate(mods)]
    got = _both(features, data)(data)
    for k, m in enumerate(mods):
        want = [(x % 2**64) % (m % 2**64) for x in data["c%d" % k].tolist()]
        assert [x % 2**64 for x in got["c%d" % k].tolist()] == want
    with pytest.raises(RuntimeError):  # 0 modulo 2^64
        FeatureEngine([Feature("c0").add_op(SelectField("c0")).add_op(Mod(2**64))])(data)


@pytest.mark.parametrize("rows", [0, 1, 1023, 1025, 8192, 8193, 16384, 16385])
@pytest.mark.parametrize("off_dtype", [torch.int32, torch.int64])
def test_truncations_around_the_rows_of_one_launch(rng, rows, off_dtype):
    """Up to 8192 rows a tensor are truncated by one workgroup, more in three launches."""
    from recis_amd import ops

    seqs = [(_offsets(rng, r, 12, off_dtype), k, side) for r, k, side in
            ((rows, 5, True), (max(0, rows - 1), 0, False), (rows // 2, 100, False))]
    values = [torch.from_numpy(rng.integers(0, 10**9, size=int(o[-1]))) for o, _, _ in seqs]
    vals, offs, drops, pads, _, _ = ops.fused_ragged_cutoff([v.cuda() for v in values], [o.cuda() for o, _, _ in seqs],
                                                            [k for _, k, _ in seqs], [s for _, _, s in seqs], [False] * 3)
    for t, (off, keep, left) in enumerate(seqs):
        lens = (off[1:] - off[:-1]).long()
        kept = lens.clamp(max=keep)
        want = torch.cat([torch.zeros(1, dtype=torch.int64), torch.cumsum(kept, 0)])
        assert torch.equal(offs[t].cpu().long(), want) and offs[t].dtype == off_dtype
        assert torch.equal(drops[t].cpu().long(), lens - kept) and torch.equal(pads[t].cpu().long(), keep - kept)
        start = off[:-1].long() + (lens - kept if left else 0)
        at = torch.arange(int(want[-1])) - torch.repeat_interleave(want[:-1], kept) + torch.repeat_interleave(start, kept)
        assert torch.equal(vals[t].cpu(), values[t][at])
    assert _lib.poll_device_errors() == 0


def test_offsets_out_of_range_are_reported_by_the_one_launch():
    from recis_amd import ops

    values = torch.arange(10).cuda()
    for bad in ([0, 4, 11], [-2, 3, 10], [0, 7, 3]):  # past the values, before them, decreasing (an empty row)
        off = torch.tensor(bad).cuda()
        vals, offs, *_ = ops.fused_ragged_cutoff([values], [off], [20], [False], [False])
        lens = [e - b if 0 <= b <= e <= 10 else 0 for b, e in zip(bad[:-1], bad[1:])]
        assert offs[0].cpu().tolist() == [0, lens[0], sum(lens)]
        assert _lib.poll_device_errors() == (0 if bad == [0, 7, 3] else 1)
