"""``FeatureEngine``: runs a list of features step by step, batching the same-typed ops
of one step into ONE fused HIP launch (mirror of ``recis.features.feature_engine``,
feature_engine.py:107-284, with the fused implementations of fused_op_impl.py:113-516
for Mod, Bucketize, Hash, IDMultiHash and SequenceTruncate). Features with identical op chains are computed
once and shared."""
from collections import defaultdict
from typing import Dict, List

import torch
from torch import nn

from .. import ops
from ..ragged.tensor import RaggedTensor
from .feature import Feature
from .op import (Bucketize, Hash, IDMultiHash, Mod, RaggedPadInfo, SelectField, SequenceTruncate, _values, _with_values,
                 sequence_truncate)


def _fused_mod(op_list, inputs):
    outs = ops.fused_uint64_mod([_values(x).cuda() for x in inputs], [op.mod_value for op in op_list])
    return [_with_values(x, o) for x, o in zip(inputs, outs)]


def _fused_bucketize(op_list, inputs):
    outs = ops.fused_bucketized([_values(x).cuda().float() for x in inputs], [op.boundary.cuda() for op in op_list])
    return [_with_values(x, o) for x, o in zip(inputs, outs)]


def _fused_bucketize_mod(op_list, inputs):
    """Bucketize followed by Mod of the same feature: one pass (``op_list``: (Bucketize, Mod) pairs)."""
    vals = [_values(x) for x in inputs]
    if all(v.is_cuda and v.dtype == torch.float32 for v in vals):
        # the common case needs no conversions: one call of the registered operator
        outs = ops.recis_ops().fused_bucketized_mod(vals, [b.boundary_on(v.device) for (b, _), v in zip(op_list, vals)],
                                                    [m.mod_value for _, m in op_list])
        outs = [o if v.dim() == 1 else o.view(v.shape) for o, v in zip(outs, vals)]
    else:
        outs = ops.fused_bucketized([v.cuda().float() for v in vals], [b.boundary.cuda() for b, _ in op_list],
                                    mods=[m.mod_value for _, m in op_list])
    return [_with_values(x, o) for x, o in zip(inputs, outs)]


def _fused_hash(op_list, inputs):
    results = [None] * len(inputs)
    for kind in ("farm", "murmur"):
        idx = [i for i, op in enumerate(op_list) if op.hash_type == kind]
        if not idx:
            continue
        outs = ops.fused_hash([inputs[i].values().cuda() for i in idx],
                              [inputs[i].offsets()[-1].cuda() for i in idx], kind)
        for i, o in zip(idx, outs):
            rest = [t.cuda() for t in inputs[i].offsets()[:-1]]
            if not rest:
                import torch
                rest = [torch.arange(o.numel() + 1, device=o.device)]
            results[i] = RaggedTensor(o, rest, None)
    return results


def _fused_multi_hash(op_list, inputs):
    outs = ops.fused_multi_hash([_values(x).cuda() for x in inputs], [op.muls for op in op_list],
                                [op.primes for op in op_list], [op.num_buckets for op in op_list])
    results, k = [], 0
    for op, x in zip(op_list, inputs):
        n = len(op.muls)
        results.append({"%s_%d" % (op.prefix, j): _with_values(x, outs[k + j]) for j in range(n)})
        k += n
    return results


_CHAIN = "bucketize+mod"   # a Bucketize whose feature goes on with a Mod: both in one launch
_FUSED = {Mod: _fused_mod, Bucketize: _fused_bucketize, Hash: _fused_hash, IDMultiHash: _fused_multi_hash,
          SequenceTruncate: sequence_truncate, _CHAIN: _fused_bucketize_mod}


def _int64s(values):
    """Moduli as the operators hand them to the kernels, modulo 2^64: they may be any uint64."""
    if not values or (max(values) < 2**63 and min(values) >= -2**63):
        return values
    return [(v + 2**63) % 2**64 - 2**63 for v in values]


class _Chains:
    """The features of an engine whose operators are all of the forms that ``feature_chains`` runs in one call: a selected
    field, then one of Hash, Mod, Bucketize + Mod, IDMultiHash or nothing, the ids possibly truncated. (31 features, batch 8192:
    331 us operator by operator, 109 in one call with three launches.)"""

    _HEADS = {(): None, (Hash,): "hash", (Mod,): "mod", (Bucketize, Mod): "bucket", (IDMultiHash,): "multi"}

    @classmethod
    def of(cls, features):
        """None when some feature has another form, or none has an operator."""
        self = cls()
        self.names, self.selects, self.hooks = [], [], []
        self.hash, self.mod, self.bucket, self.multi, self.cut = [], [], [], [], []  # (place of the feature, its op(s))
        self.first = None  # the first feature with an operator
        for place, f in enumerate(features):
            ops_of = f.ops
            kinds = tuple(type(op) for op in ops_of)
            if not kinds or kinds[0] is not SelectField:
                return None
            cut = kinds[-1] is SequenceTruncate
            head = kinds[1:-1] if cut else kinds[1:]
            if head not in cls._HEADS or (cut and head in ((Bucketize, Mod), (IDMultiHash,))):
                return None
            self.names.append(f.name)
            self.selects.append(ops_of[0])
            for op in ops_of:
                self.hooks += [op._forward_hooks, op._forward_pre_hooks]
            kind = cls._HEADS[head]
            if kind == "bucket":
                self.bucket.append((place, ops_of[1], ops_of[2]))
            elif kind is not None:
                getattr(self, kind).append((place, ops_of[1]))
            if cut:
                self.cut.append((place, ops_of[-1]))
            if len(kinds) > 1 and self.first is None:
                self.first = place
        return None if self.first is None else self

    def run(self, data):
        """The results of the features in order, or None: something asks for the operators one by one."""
        if any(self.hooks):
            return None
        for _, op in self.cut:
            if op.check_length or not op.truncate or op.n_dims != 2:
                return None
        xs = [data[op._name] if op._from_dict else data for op in self.selects]
        vals = [x._values if type(x) is RaggedTensor else x for x in xs]
        for v in vals:
            if type(v) is not torch.Tensor:
                return None
        if not vals[self.first].is_cuda:
            return None
        for place, _ in self.hash:
            x = xs[place]
            if type(x) is not RaggedTensor or len(x._offsets) < 2 or not all(o.is_cuda for o in x._offsets):
                return None
        hash_at = {place: k for k, (place, _) in enumerate(self.hash)}
        n_hash = len(self.hash)
        mod_at = {place: n_hash + k for k, (place, _) in enumerate(self.mod)}
        direct, cut_from, cut_offsets = [], [], []
        for place, op in self.cut:
            x = xs[place]
            if type(x) is not RaggedTensor:
                return None
            at = hash_at.get(place, mod_at.get(place))
            if at is None:
                direct.append(vals[place])
                at = -len(direct)
            cut_from.append(at)
            cut_offsets.append(x._offsets[-2 if place in hash_at else -1])
        outs = ops.recis_ops().feature_chains(
            [vals[p] for p, _ in self.hash], [xs[p]._offsets[-1] for p, _ in self.hash],
            [1 if op.hash_type == "murmur" else 0 for _, op in self.hash],
            [vals[p] for p, _ in self.mod], _int64s([op.mod_value for _, op in self.mod]),
            [vals[p] for p, _, _ in self.bucket], [b.boundary_on(vals[p].device) for p, b, _ in self.bucket],
            [m.mod_value for _, _, m in self.bucket],
            [vals[p] for p, _ in self.multi], [len(op.muls) for _, op in self.multi],
            [v for _, op in self.multi for v in op.muls], [v for _, op in self.multi for v in op.primes],
            [v for _, op in self.multi for v in op.num_buckets],
            direct, cut_from, cut_offsets, [op.seq_len for _, op in self.cut],
            [op.truncate_side == "left" for _, op in self.cut])
        if not outs:
            return None
        results = xs
        k = n_hash + len(self.mod)
        for place, _, _ in self.bucket:
            results[place] = _with_values(xs[place], outs[k])
            k += 1
        for place, op in self.multi:
            x, n = xs[place], len(op.muls)
            results[place] = {"%s_%d" % (op.prefix, j): _with_values(x, outs[k + j]) for j in range(n)}
            k += n
        n_cut = len(self.cut)
        for j, (place, op) in enumerate(self.cut):
            x = xs[place]
            if place in hash_at:
                rest = x._offsets[:-1]
                shape, weight = [rest[0].numel() - 1] + [-1] * len(rest), None
                del hash_at[place]
            else:
                shape, weight = list(x.dense_shape), x.weight()
                mod_at.pop(place, None)
            shape[1] = op.seq_len
            values, offsets, drops, pads, drop_side, pad_side = outs[k + j::n_cut][:6]
            results[place] = RaggedTensor(values, [offsets], weight, shape)
            results[place].set_pad_info(RaggedPadInfo(drops, pads, drop_side, pad_side))
        for place, at in hash_at.items():
            results[place] = RaggedTensor(outs[at], xs[place]._offsets[:-1], None)
        for place, at in mod_at.items():
            results[place] = _with_values(xs[place], outs[at])
        return results


class FeatureEngine(nn.Module):
    def __init__(self, feature_list: List[Feature]):
        super().__init__()
        self._features = nn.ModuleDict()
        self._alias = {}
        by_hash = defaultdict(list)
        for f in feature_list:
            by_hash[f.get_hash()].append(f)
        for group in by_hash.values():
            primary = group[0]
            if primary.name in self._features:
                raise ValueError("Duplicate feature name: %s" % primary.name)
            if primary.compiled:
                raise ValueError("feature %s has been compiled" % primary.name)
            primary.compiled_(True)
            self._features[primary.name] = primary
            for dup in group[1:]:
                self._alias[dup.name] = primary.name
        # step k = the k-th op of every feature that has one, grouped by op class
        self._steps = []
        feats = list(self._features.values())
        self._chains = _Chains.of(feats)
        depth = max((len(f.ops) for f in feats), default=0)
        done_early = set()  # (feature, k): op k of the feature was applied together with op k - 1
        for k in range(depth):
            groups = defaultdict(list)
            for f in feats:
                if k < len(f.ops) and (f.name, k) not in done_early:
                    op = f.ops[k]
                    nxt = f.ops[k + 1] if k + 1 < len(f.ops) else None
                    if type(op) is Bucketize and type(nxt) is Mod and 0 < nxt.mod_value and \
                            not (nxt._forward_hooks or nxt._forward_pre_hooks or op._forward_hooks or op._forward_pre_hooks):
                        groups[_CHAIN].append((f.name, (op, nxt)))
                        done_early.add((f.name, k + 1))
                        continue
                    groups[type(op) if type(op) in _FUSED else ("single", f.name)].append((f.name, op))
            self._steps.append(groups)

    def forward(self, data: Dict, remain_no_use_data: bool = True) -> Dict:
        assert isinstance(data, dict), "data must be a dict"
        chains = self.__dict__.get("_chains")
        found = chains.run(data) if chains is not None else None
        state = dict(zip(chains.names, found)) if found is not None else {}
        for step_idx, groups in enumerate(self._steps if found is None else ()):
            for key, members in groups.items():
                names = [n for n, _ in members]
                op_list = [op for _, op in members]
                inputs = [state[n] if step_idx > 0 else data for n in names]
                if key in _FUSED and (len(members) > 1 or key == _CHAIN):
                    outs = _FUSED[key](op_list, inputs)
                else:
                    # Module.__call__ costs several microseconds of hook bookkeeping per op, which is
                    # most of a SelectField; ops with no hooks registered are called directly
                    outs = [op(x) if (op._forward_hooks or op._forward_pre_hooks) else op.forward(x)
                            for op, x in zip(op_list, inputs)]
                for n, o in zip(names, outs):
                    state[n] = o
        results = dict(data) if remain_no_use_data else {}
        for name, out in state.items():
            if isinstance(out, dict):
                results.update(out)
            else:
                results[name] = out
        for dup, primary in self._alias.items():
            results[dup] = results[primary]
        return results
