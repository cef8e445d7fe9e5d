"""``EmbeddingOption`` and ``DynamicEmbedding``: the mirror of
``recis.nn.modules.embedding`` (embedding.py:161-624) for one GPU that owns the whole
table (world size 1: the id / row / gradient all-to-alls of the reference are the
identity and are left out)."""
import json
import math
import os
from dataclasses import dataclass, field
from typing import List, Optional, Union

import torch

from ... import ops
from ...ragged.tensor import RaggedTensor
from ..functional.embedding_ops import ragged_embedding_segment_reduce
from ..hashtable_hook import AdmitHook, FilterHook
from ..initializers import ConstantInitializer, Initializer
from .hashtable import (GradIDMeanFunction, HashTable, HashTableLookupHelpFunction, accept_planned_grad, gen_slice,
                        pools_readonly)


class _Done:
    """Stands where the reference keeps the handle of an asynchronous all-to-all: with one GPU
    there is nothing to wait for."""

    def wait(self):
        return None


@dataclass
class ExchangeIDsResults:
    """embedding.py:121-140, for one GPU: ``ids`` are the distinct ids of the batch (what the
    reference receives from its peers), ``parts`` / ``parts_reverse`` their count, ``plan`` the
    batch plan the later stages reuse."""

    ids: torch.Tensor
    ids_await: object
    parts: List[int]
    parts_reverse: List[int]
    reverse_index: torch.Tensor
    offsets: torch.Tensor
    plan: object = None


@dataclass
class ExchangeEmbResults:
    """embedding.py:142-158."""

    emb: torch.Tensor
    reverse_index: torch.Tensor
    emb_shape: List[int]
    offsets: torch.Tensor
    emb_await: Optional[object] = None
    plan: object = None


@dataclass
class EmbeddingOption:
    embedding_dim: int = 16
    block_size: int = 10240
    dtype: torch.dtype = torch.float32
    device: torch.device = torch.device("cuda")
    trainable: bool = True
    pg: object = None
    max_partition_num: int = 65536
    shared_name: str = "embedding"
    children: List[str] = field(default_factory=list)
    coalesced: Optional[bool] = False
    initializer: Optional[Initializer] = None
    use_weight: Optional[bool] = True
    combiner: Optional[str] = "sum"
    combiner_kwargs: Optional[dict] = None
    grad_reduce_by: Optional[str] = "worker"
    filter_hook: Optional[FilterHook] = None
    admit_hook: Optional[AdmitHook] = None
    fp16_enabled: bool = False
    reserve_rows: int = 0  # addition: pre-size the map and the row storage

    def __post_init__(self):
        if not self.children:
            self.children = [self.shared_name]
        if self.initializer is None:
            self.initializer = ConstantInitializer(init_val=0)
        if self.fp16_enabled:
            assert self.dtype in (torch.int8,), "only int8 emb can set fp16_enabled"
        assert self.combiner in ["sum", "mean", "tile", "max"], \
            "Hashtable combiner only support [sum/mean/tile/max], but got %s" % self.combiner
        if self.combiner == "tile":
            if self.combiner_kwargs is None:
                raise RuntimeError("combiner_kwargs must be set when combiner is tile.")
            if "tile_len" not in self.combiner_kwargs:
                raise RuntimeError("tile_len must be in combiner_kwargs when combiner is tile.")

    def coalesced_info(self):
        return json.dumps({
            "dim": self.embedding_dim, "dtype": str(self.dtype), "device": str(torch.device(self.device).type),
            "initializer": str(self.initializer), "grad_reduce_by": self.grad_reduce_by,
            "filter_hook": str(self.filter_hook),
        })

    def runtime_info(self):
        return json.dumps({
            "combiner": self.combiner, "use_weight": self.use_weight, "trainable": self.trainable,
            "admit_hook": str(self.admit_hook), "fp16_enabled": self.fp16_enabled,
        })


def lookup_unique_rows(hashtable: HashTable, unique_ids, admit_hook=None, trainable=True, grad_key=None):
    """Rows of ids that are already unique: the lookup autograd function, the
    last-seen-step stamp, no second dedup. ``grad_key``: see ``HashtableImpl.accept_grad``."""
    from .hashtable_hook_impl import HashtableHookFactory

    impl = hashtable._hashtable_impl
    float_table = hashtable._dtype not in (torch.int8, torch.int32, torch.int64)
    if hashtable.training and trainable and float_table:
        admit_impl = HashtableHookFactory().create_admit_hook(hashtable, admit_hook) if admit_hook else None
        emb_idx, emb = HashTableLookupHelpFunction.apply(unique_ids, impl, hashtable._backward_holder, admit_impl,
                                                         grad_key)
        hashtable._filter_hook_impl(emb_idx)
        return emb
    readonly = (not hashtable.training) or admit_hook is not None or not float_table
    _, emb = impl.embedding_lookup(unique_ids.detach(), readonly)
    if hashtable.training and not readonly:
        hashtable._filter_hook_impl(_)
    return emb


class LookupPoolFunction(torch.autograd.Function):
    """Read-only lookup (an admit hook keeps new keys out) of a plan's unique ids in training and sum / mean pooling
    straight out of the table: the ``[U, D]`` copy of the looked-up rows (lookup function +
    ``ragged_embedding_segment_reduce``, recis/nn/modules/embedding.py:592-624) is never made. Backward hands the
    pooled gradients to the table unsummed; keys the table does not hold carry a negative index and take none. (The
    lookup that admits keys is ``HashtableImpl.lookup_train``.)"""

    @staticmethod
    def forward(ctx, backward_holder, impl, plan, weight, offsets, combiner, unit_segments=False, split=None):
        """``unit_segments``: one id per segment (sum == mean == the row itself), so every unique row is read once and
        written to its occurrences. ``split``: row counts to cut the pooled output into (one part per feature of a group that is pooled
        in one go); the parts are returned as separate outputs, views of the one buffer, and backward takes
        their gradients as they come: slices of one buffer are used in place, anything else is concatenated."""
        index = impl.lookup_index(plan.unique, True)
        if unit_segments:
            out = impl.expand_rows(plan, index, weight, None, None)
        else:
            chunks, chunk_rows = impl.emb_blocks()
            out = ops.segment_reduce_forward_blocks(chunks, chunk_rows, index, weight, plan.inverse, offsets, combiner)
        ctx.impl, ctx.plan, ctx.combiner, ctx.unit_segments = impl, plan, combiner, unit_segments
        ctx.split, ctx.out_shape, ctx.out_dtype = split, tuple(out.shape), out.dtype
        ctx.save_for_backward(index, weight, offsets)
        ctx.set_materialize_grads(False)
        ctx.mark_non_differentiable(index)
        return (index,) + (tuple(torch.split(out, split)) if split is not None else (out,))

    @staticmethod
    def backward(ctx, _grad_index, *grads):
        index, weight, offsets = ctx.saved_tensors
        if all(g is None for g in grads):  # a function behind the outputs returned none: zeros, which still are a gradient
            grads = (torch.zeros(ctx.out_shape if ctx.split is None else (ctx.split[0], ctx.out_shape[1]), dtype=ctx.out_dtype,
                                 device=offsets.device),) + grads[1:]
        grad = grads[0] if ctx.split is None else _joined(grads, ctx.split, ctx.out_shape)
        # sum / mean: the gradient of a unique row is a gather-reduce over its occurrence list; it is handed
        # over unsummed, so that the optimizer step can sum and update the row in one launch
        if ctx.unit_segments and weight is None:
            src, coef = ctx.plan.occ, None  # an occurrence is its own segment
        else:
            src, coef = ctx.plan.src_coef_for_pool(offsets.contiguous(), weight, ctx.combiner == "mean")
        accept_planned_grad(ctx.impl, index, ctx.plan, grad.contiguous(), src, coef, may_miss=True)
        return (None,) * 8


def _joined(grads, split, shape):
    """The gradients of the parts of one pooled output as one ``shape`` tensor: in place when they are
    consecutive slices of one buffer (what a caller that keeps its gradients in one array hands over),
    concatenated otherwise (a missing gradient counts as zeros)."""
    like = next(g for g in grads if g is not None)
    first = grads[0]
    if first is not None and first.is_contiguous():
        at = first.data_ptr()
        for g, rows in zip(grads, split):
            if g is None or g.dtype != first.dtype or not g.is_contiguous() or g.data_ptr() != at \
                    or g.untyped_storage().data_ptr() != first.untyped_storage().data_ptr():
                break
            at += rows * shape[1] * g.element_size()
        else:
            whole = torch.as_strided(first, shape, (shape[1], 1), first.storage_offset())
            return whole
    return torch.cat([g if g is not None else like.new_zeros((rows, shape[1])) for g, rows in zip(grads, split)])


def _pools_out_of_the_table(hashtable, opt, n_occ, n_offsets):
    """Whether lookup_and_pool takes the path that pools straight out of the table rows."""
    float_table = hashtable._dtype in (torch.float32, torch.bfloat16, torch.float16)
    sparse_mean = opt.combiner == "mean" and not n_occ / n_offsets > 5
    id_mean = opt.grad_reduce_by == "id" and hashtable.training and opt.trainable
    return opt.combiner in ("sum", "mean") and float_table and not sparse_mean and not id_mean


def lookup_and_pool(hashtable: HashTable, plan, weight, offsets, opt, unit_segments=False, combiner_kwargs=None,
                    split=None):
    """Rows of the plan's unique ids pooled per segment, for what ``HashtableImpl.lookup_train`` and
    ``lookup_pool_readonly`` leave over. Under an admit hook sum / mean over a float table go through
    ``LookupPoolFunction`` (pooling reads the table directly); everything else looks the rows up first and pools the
    copy. ``unit_segments``: ``offsets`` are 0, 1, 2, ... (dense ``[B, 1]`` id tensors). ``split``: return the pooled
    rows cut into parts of these row counts (a tuple)."""
    id_mean = opt.grad_reduce_by == "id" and hashtable.training and opt.trainable
    if _pools_out_of_the_table(hashtable, opt, plan.n, offsets.numel()):
        impl = hashtable._hashtable_impl
        if weight is not None and weight.dtype != hashtable._dtype:
            weight = weight.to(hashtable._dtype)
        if hashtable.training and opt.trainable:  # under an admit hook, or lookup_train would have taken it
            from .hashtable_hook_impl import HashtableHookFactory, ReadOnlyHookImpl
            admit = HashtableHookFactory().create_admit_hook(hashtable, opt.admit_hook)
            assert isinstance(admit, ReadOnlyHookImpl), "admit hook only support ReadOnlyHook yet, but got: %s" % admit
            index, *outs = LookupPoolFunction.apply(hashtable._backward_holder, impl, plan, weight, offsets,
                                                    opt.combiner, unit_segments, split)
            hashtable._filter_hook_impl(index)
            return outs[0] if split is None else tuple(outs)
        readonly = (not hashtable.training) or opt.admit_hook is not None
        index = impl.lookup_index(plan.unique.detach(), readonly)
        if hashtable.training and not readonly:
            hashtable._filter_hook_impl(index)
        chunks, chunk_rows = impl.emb_blocks()
        out = ops.segment_reduce_forward_blocks(chunks, chunk_rows, index, weight, plan.inverse, offsets,
                                                opt.combiner)
        return out if split is None else torch.split(out, split)
    emb = lookup_unique_rows(hashtable, plan.unique, opt.admit_hook, opt.trainable)
    inverse = plan.inverse
    if id_mean:
        # mean over the duplicates of each id: pool the expanded rows instead
        emb = GradIDMeanFunction.apply(emb, inverse, plan)
        inverse, plan = None, None
    if weight is not None and weight.dtype != emb.dtype:
        weight = weight.to(emb.dtype)
    out = ragged_embedding_segment_reduce(emb, weight, inverse, offsets, opt.combiner,
                                          combiner_kwargs if combiner_kwargs is not None else opt.combiner_kwargs,
                                          plan=plan)
    return out if split is None else torch.split(out, split)


class DynamicEmbedding(torch.nn.Module):
    def __init__(self, emb_opt: EmbeddingOption, pg=None):
        super().__init__()
        self._emb_opt = emb_opt
        self._world_size = int(os.environ.get("WORLD_SIZE", 1))
        self._rank = int(os.environ.get("RANK", 0))
        if self._world_size != 1:
            raise NotImplementedError("this build runs one GPU that owns the whole table (WORLD_SIZE=1)")
        self._hashtable = HashTable(
            embedding_shape=[emb_opt.embedding_dim], block_size=emb_opt.block_size, dtype=emb_opt.dtype,
            device=emb_opt.device, initializer=emb_opt.initializer, children=emb_opt.children,
            name=emb_opt.shared_name, coalesced=emb_opt.coalesced,
            slice=gen_slice(shard_index=self._rank, shard_num=self._world_size),
            grad_reduce_by=emb_opt.grad_reduce_by, filter_hook=emb_opt.filter_hook,
            reserve_rows=emb_opt.reserve_rows)

    def deal_with_tensor(self, input_tensor: Union[torch.Tensor, RaggedTensor]):
        if isinstance(input_tensor, RaggedTensor):
            val = input_tensor.values()
            weight = input_tensor.weight()
            offsets = input_tensor.offsets()[-1]
            shape = input_tensor.real_shape(0, -1)
            if not math.prod(shape) == (offsets.numel() - 1):
                raise RuntimeError("RaggedTensor must pad before lookup, got: %s" % input_tensor)
        elif isinstance(input_tensor, torch.Tensor):
            if input_tensor.is_sparse:
                raise TypeError("RaggedDynamicEmbedding doesn't support sparse ids")
            val = input_tensor.reshape(-1)
            bs, fea_dim = input_tensor.shape[0], input_tensor.shape[1]
            offsets = torch.arange(bs + 1, device=val.device) * fea_dim
            weight = None
            shape = tuple(input_tensor.shape[:-1])
        else:
            raise TypeError("DynamicEmbedding only support RaggedTensor or dense tensor, got %s" % type(input_tensor))
        return val, offsets, weight, shape

    def forward(self, input_ids, input_weights=None):
        opt = self._emb_opt
        val, offsets, weight, shape = self.deal_with_tensor(input_ids)
        dev = self._hashtable._impl_device
        val, offsets = val.to(dev), offsets.to(dev)
        if input_weights is not None:
            weight = input_weights
        if weight is not None:
            weight = weight.to(dev) if opt.use_weight else None
        out = self._pooled(val, offsets, weight, input_ids.shape[1] if type(input_ids) is torch.Tensor and input_ids.dim() == 2 else None)
        if opt.combiner == "tile":
            return out.view(tuple(shape) + (opt.combiner_kwargs["tile_len"] * opt.embedding_dim,))
        return out.view(tuple(shape) + (opt.embedding_dim,))

    def _pooled(self, val, offsets, weight, width):
        """The rows of ``val`` pooled per segment: in one native call where the table, the combiner and the mode
        allow it. ``width`` ids per segment when the ids were a dense tensor."""
        opt, table = self._emb_opt, self._hashtable
        if table._dtype in (torch.float32, torch.bfloat16, torch.float16) and opt.combiner in ("sum", "mean"):
            ids, offs = (val, offsets) if not width or weight is not None else (val.view(-1, width), None)
            if not table.training and val.dtype == torch.int64 and pools_readonly(table):
                return table._hashtable_impl.lookup_pool_readonly([ids], [offs], [weight], None, opt.combiner == "mean")[0]
            if table.training and opt.trainable and opt.admit_hook is None and opt.grad_reduce_by != "id":
                res = table._hashtable_impl.lookup_train([ids], [offs], [weight], None, opt.combiner, [], True, None, None)
                if res is not None:
                    if not isinstance(table._filter_hook_impl, torch.nn.Identity):
                        table._filter_hook_impl(res[3][: res[1].U])
                    return res[0][0]
        plan = ops.ids_unique_plan(val, wait=False, need_pos=False)
        return lookup_and_pool(table, plan, weight, offsets, opt)

    # The staged form of forward (embedding.py:498-624), which EmbeddingEngine-style callers drive
    # stage by stage. With one GPU the two all-to-alls are the identity: exchange_ids is the dedup,
    # lookup_exchange_emb the table lookup of the distinct ids, emb_reduce the pooling. forward()
    # above fuses the last two (pooling reads the table rows directly).
    def exchange_ids(self, ids: torch.Tensor, offsets: torch.Tensor):
        plan = ops.ids_unique_plan(ids, wait=True, need_pos=False)
        n = int(plan.U)
        return ExchangeIDsResults(ids=plan.unique, ids_await=_Done(), parts=[n], parts_reverse=[n],
                                  reverse_index=plan.inverse, offsets=offsets, plan=plan)

    def lookup_exchange_emb(self, ids_exchange_result: ExchangeIDsResults, admit_hook=None):
        ids_exchange_result.ids_await.wait()
        emb = lookup_unique_rows(self._hashtable, ids_exchange_result.ids, admit_hook, self._emb_opt.trainable)
        return ExchangeEmbResults(emb=emb, emb_await=_Done(), reverse_index=ids_exchange_result.reverse_index,
                                  emb_shape=list(emb.shape), offsets=ids_exchange_result.offsets,
                                  plan=ids_exchange_result.plan)

    def wait_exchange_emb(self, emb_exchange_result: ExchangeEmbResults):
        emb_exchange_result.emb_await.wait()
        return emb_exchange_result.emb.view(emb_exchange_result.emb_shape)

    def emb_reduce(self, emb_exchange_result: ExchangeEmbResults, weight, combiner, combiner_kwargs,
                   fp16_enable=False):
        emb = self.wait_exchange_emb(emb_exchange_result)
        if emb.dtype in (torch.int8,):
            emb = emb.to(torch.float16 if fp16_enable else torch.float32)
        if weight is not None and weight.dtype != emb.dtype:
            weight = weight.to(emb.dtype)
        return ragged_embedding_segment_reduce(emb, weight, emb_exchange_result.reverse_index,
                                               emb_exchange_result.offsets, combiner, combiner_kwargs,
                                               plan=emb_exchange_result.plan)

    @property
    def hashtable(self):
        return self._hashtable
