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
