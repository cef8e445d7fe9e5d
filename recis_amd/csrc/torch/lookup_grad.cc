// The training lookups of the module layer with their autograd nodes: what EmbeddingEngine and
// HashTable call once per table and step (recis/nn/modules/embedding_engine.py:607-675,
// recis/nn/modules/hashtable.py:425-586). The forward queues dedup + lookup + pooling without waiting
// for the device. The node's backward hands the gradients to the table unsummed; the batch's unique count, and what
// the plan's kernels reported with it, is read there, behind the forward's launches: it has arrived or is about to, and
// a plan that dropped entries raises before its gradient has reached the table. Nothing per feature is left to Python (a node written in Python costs 2 us per output each way: with 39
// features that was most of a small step).
#include <torch/csrc/autograd/custom_function.h>
#include <torch/csrc/autograd/function.h>
#include <torch/csrc/autograd/functions/utils.h>
#include <torch/csrc/autograd/saved_variable.h>

#include <algorithm>

#include "abi_util.h"
#include "ops.h"
#include "table.h"

using recis::BatchPlanPtr;
using recis::hipabi::block_ptr_table;
using recis::hipabi::check;
using recis::hipabi::dtype_code;
using recis::hipabi::index_kind;
using recis::hipabi::part_of;
using recis::hipabi::stream_of;
using recis::hipabi::TensorOrNone;

namespace {

using torch::autograd::SavedVariable;

// The backward of one lookup of a table: the parts' gradients go to the table as they come.
struct LookupBackward : public torch::autograd::Node {
  c10::intrusive_ptr<Hashtable> table;
  BatchPlanPtr plan;
  SavedVariable saved_index;
  std::vector<int64_t> split;        // rows per output
  std::vector<int64_t> first_shape;  // of the first output
  // Pooled segments; both undefined: one id per segment. They may be the caller's own tensors: saved as any node saves its
  // inputs, so that a buffer refilled before the backward is refused and saved-tensor hooks see them.
  SavedVariable saved_offsets, saved_weight;
  at::Tensor occ;                    // what the pooling noted per occurrence, or undefined
  bool mean = false;
  std::vector<int64_t> batch, seq;   // padded outputs (tile): samples and rows per sample of each
  bool tile = false;
  bool columns = false;              // one id per sample, of a plan that no other lookup shares

  torch::autograd::variable_list apply(torch::autograd::variable_list&& grads) override {
    std::lock_guard<std::mutex> lock(mutex_);
    TORCH_CHECK(plan.defined(), torch::autograd::ERR_BACKWARD_TWICE);
    at::NoGradGuard no_grad;
    const at::Tensor index = saved_index.unpack(), offsets = saved_offsets.unpack(), weight = saved_weight.unpack();
    // Functions behind the outputs that returned no gradient: zeros, which still are one (the rows take a step of
    // their momentum). An output that is undefined beside others that are not counts as zeros anyway.
    if (!grads.empty() && std::none_of(grads.begin(), grads.end(), [](const at::Tensor& g) { return g.defined(); }))
      grads[0] = at::zeros(first_shape, at::TensorOptions().device(index.device()).dtype(table->dtype()));
    if (tile) {
      table->AcceptTileGrad(index, plan, offsets, batch, seq, grads);
      return {};
    }
    if (columns && table->AcceptColumnSlices(index, plan, grads, split)) return {};
    std::vector<TensorOrNone> parts;
    parts.reserve(grads.size());
    for (auto& g : grads) parts.push_back(g.defined() ? TensorOrNone(std::move(g)) : c10::nullopt);
    TensorOrNone src, coef;
    if (occ.defined()) {
      auto lists = plan->SrcCoefFromOcc(occ, offsets, weight.defined() || mean);
      src = std::get<0>(lists);
      coef = std::get<1>(lists);
    } else if (offsets.defined()) {
      auto lists = plan->SrcCoefForPool(offsets, weight.defined() ? TensorOrNone(weight) : c10::nullopt, mean);
      src = std::get<0>(lists);
      coef = std::get<1>(lists);
    }
    table->AcceptSplitGrad(index, plan, parts, split, src, coef, plan->serial(), /*may_miss=*/false, /*settle=*/true);
    return {};
  }
  void release_variables() override {
    std::lock_guard<std::mutex> lock(mutex_);
    plan.reset();
    saved_index.reset_data();
    saved_offsets.reset_data();
    saved_weight.reset_data();
    occ.reset();
  }
  std::string name() const override { return "RecisLookupBackward"; }
};

// Whether the pooling notes segment and coefficient of every occurrence for the backward (recis_csr_lists_from_occ), or
// the backward searches the offsets (recis_csr_fill_lists). The notes cost a write and one scattered 8-byte read an entry,
// whatever the segments; up to half a million entries (4 MB of notes, an XCD's L2) that is always the cheaper. Beyond it the
// reads miss the L2, and what the search costs depends on the offsets beyond its table of 2048 in LDS: few when segments are
// long. Measured, us (search - notes with their writing; power-law ids), per ids of a segment on average:
//   unweighted          8     30    100    400        weighted     8     30    100    400
//   0.26 M            7.6    6.4    4.6    3.3                   8.4    7.1    5.4    4.0
//   0.52 M            8.8    4.8    4.0    2.1                   9.9    6.2    4.7    3.1
//   0.79 M            8.5    1.3   -1.7   -2.8                  11.6    4.5    1.4   -0.8
//   1.05 M           11.2    2.6   -4.3   -5.4                  15.6    8.1    1.9   -0.9
//   2.10 M           23.8    8.9  -13.2  -19.8                  36.3   21.4    2.7   -7.6
bool NotesOccurrences(int64_t n, int64_t segments, bool weighted) {
  if (n == 0 || segments == 0) return false;
  return n <= (int64_t(1) << 19) || n <= (weighted ? 128 : 32) * segments;
}

// The outputs of a lookup, with the node behind them (none when gradients are not recorded).
std::vector<at::Tensor> outputs_of(const at::Tensor& whole, const std::vector<std::vector<int64_t>>& shapes,
                                   const std::vector<int64_t>& split, const std::shared_ptr<LookupBackward>& node) {
  std::vector<at::Tensor> out;
  out.reserve(split.size());
  int64_t first = 0;
  for (size_t k = 0; k < split.size(); ++k) {
    out.push_back(part_of(whole, first * whole.size(1), shapes[k]));
    first += split[k];
  }
  if (node) {
    for (auto& o : out) torch::autograd::set_history(o, node);
  }
  return out;
}

}  // namespace

c10::optional<std::vector<at::Tensor>> Hashtable::DenseLookupTrain(const std::vector<at::Tensor>& cols,
                                                                   const c10::optional<std::vector<int64_t>>& tags,
                                                                   const c10::optional<std::string>& stamp_slot,
                                                                   const c10::optional<at::Tensor>& stamp_value) {
  auto found = DenseLookupExpand(cols, tags, stamp_slot, stamp_value);
  if (!found.has_value()) return c10::nullopt;
  const at::Tensor& out = std::get<2>(*found);
  std::vector<std::vector<int64_t>> shapes;
  std::vector<int64_t> split;
  for (const auto& c : cols) {
    split.push_back(c.size(0));
    shapes.push_back({c.size(0), out.size(1)});
  }
  std::shared_ptr<LookupBackward> node;
  if (at::GradMode::is_enabled()) {
    node = std::make_shared<LookupBackward>();
    node->table = c10::intrusive_ptr<Hashtable>::reclaim_copy(this);
    node->plan = std::get<0>(*found);
    node->saved_index = SavedVariable(std::get<1>(*found), false);
    node->split = split;
    node->first_shape = shapes[0];
    node->columns = true;
  }
  return outputs_of(out, shapes, split, node);
}

// Segments of several features as one list: the given offsets, and 0, width, 2 * width, ... for the dense
// tensors (undefined entries). int32.
at::Tensor Hashtable::GroupOffsets(const std::vector<TensorOrNone>& offsets, const std::vector<int64_t>& segments,
                                   const std::vector<int64_t>& widths, const std::vector<int64_t>& n_ids) const {
  auto i32 = at::TensorOptions().device(device_).dtype(at::kInt);
  std::vector<at::Tensor> keep;  // alive until the launch is queued
  std::vector<const int32_t*> ptrs(offsets.size(), nullptr);
  int64_t total = 1;
  for (size_t k = 0; k < offsets.size(); ++k) {
    total += segments[k];
    if (!offsets[k].has_value() || !offsets[k]->defined()) continue;
    keep.push_back(offsets[k]->to(i32).contiguous());
    ptrs[k] = keep.back().data_ptr<int32_t>();
  }
  if (offsets.size() == 1 && !keep.empty()) return keep[0];
  at::Tensor out = at::empty({total}, i32);
  check(recis_group_offsets(ptrs.data(), segments.data(), widths.data(), n_ids.data(), static_cast<int64_t>(offsets.size()),
                            out.data_ptr<int32_t>(), stream_of(device_)));
  return out;
}

c10::optional<std::tuple<std::vector<at::Tensor>, BatchPlanPtr, TensorOrNone, at::Tensor>> Hashtable::LookupTrain(
    const std::vector<at::Tensor>& values, const std::vector<TensorOrNone>& offsets,
    const std::vector<TensorOrNone>& weights, const c10::optional<std::vector<int64_t>>& tags,
    const std::string& combiner, const std::vector<int64_t>& tile_len, bool lean,
    const c10::optional<BatchPlanPtr>& shared_plan, const c10::optional<at::Tensor>& shared_offsets) {
  const size_t n = values.size();
  TORCH_CHECK(n > 0 && offsets.size() == n && weights.size() == n, "lookup_train: one entry per feature in every list");
  TORCH_CHECK(combiner == "sum" || combiner == "mean" || combiner == "tile", "lookup_train: combiner ", combiner);
  const bool tile = combiner == "tile", mean = combiner == "mean";
  TORCH_CHECK(!tile || tile_len.size() == n, "lookup_train: one tile_len per feature");
  c10::DeviceGuard guard(device_);
  std::vector<at::Tensor> ids;
  std::vector<int64_t> segments(n), widths(n), n_ids(n);
  ids.reserve(n);
  bool unit = true, any_weight = false;
  int64_t total_ids = 0, total_segments = 0;
  for (size_t k = 0; k < n; ++k) {
    const at::Tensor& v = values[k];
    const bool as_is = v.device() == device_ && v.scalar_type() == at::kLong && v.is_contiguous();
    ids.push_back((as_is ? v : v.to(at::TensorOptions().device(device_).dtype(at::kLong)).contiguous()).view({-1}));
    n_ids[k] = ids[k].numel();
    if (offsets[k].has_value() && offsets[k]->defined()) {
      segments[k] = offsets[k]->numel() - 1;
      unit = false;
    } else {
      widths[k] = DenseWidth(v);
      segments[k] = n_ids[k] / widths[k];
      unit = unit && widths[k] == 1;
    }
    any_weight = any_weight || (weights[k].has_value() && weights[k]->defined());
    total_ids += n_ids[k];
    total_segments += segments[k];
  }
  // few ids per segment: "mean" divides by the sum of the weights (embedding_ops.py:332-420), another path
  if (mean && !(static_cast<double>(total_ids) / static_cast<double>(total_segments + 1) > 5)) return c10::nullopt;
  const bool unit_path = unit && !tile;

  BatchPlanPtr plan;
  at::Tensor merged;
  if (shared_plan.has_value() && shared_plan->defined()) {
    plan = *shared_plan;
    merged = shared_offsets.has_value() ? *shared_offsets : at::Tensor();
  } else {
    plan = PlanLookup(ids, tags, /*wait=*/false, /*need_inverse=*/!(unit_path && lean), /*need_pos=*/false);
  }
  if (!merged.defined() && !unit_path) merged = GroupOffsets(offsets, segments, widths, n_ids);
  c10::optional<at::Tensor> found = PlanIndex(plan);
  at::Tensor index = found.has_value() ? *found : LookupIndexCounted(plan, true);

  const bool recorded = at::GradMode::is_enabled();
  auto emb = slot_group_->EmbSlot();
  const auto& chunks = emb->Chunks();
  const int64_t D = emb->FlatSize();
  std::vector<std::vector<int64_t>> shapes(n);
  std::vector<int64_t> split = segments;
  at::Tensor out, weight, occ, back_offsets = merged;
  if (tile) {
    int64_t rows = 0;
    for (size_t k = 0; k < n; ++k) rows += segments[k] * tile_len[k];
    out = at::empty({rows, D}, at::TensorOptions().device(device_).dtype(dtype_));
    at::Tensor rev = plan->inverse(), table = block_ptr_table(chunks);
    check(recis_ragged_tile_blocks(segments.data(), tile_len.data(), static_cast<int64_t>(n), rev.data_ptr(), 0, plan->n(),
                                   merged.data_ptr(), index_kind(merged, "offsets"),
                                   reinterpret_cast<const void* const*>(table.data_ptr()), static_cast<int64_t>(chunks.size()),
                                   emb->ChunkRows(), chunks.empty() ? 0 : recis::hipabi::row_pitch_bytes(chunks[0]),
                                   index.data_ptr<int64_t>(), index.numel(), dtype_code(dtype_), out.data_ptr(), D, stream_of(device_)));
    for (size_t k = 0; k < n; ++k) {
      split[k] = segments[k] * tile_len[k];
      shapes[k] = {segments[k], tile_len[k] * D};
    }
  } else {
    if (any_weight) {
      std::vector<at::Tensor> parts;
      auto opt = at::TensorOptions().device(device_).dtype(dtype_);
      for (size_t k = 0; k < n; ++k) {
        const bool has = weights[k].has_value() && weights[k]->defined();
        TORCH_CHECK(!has || weights[k]->numel() == n_ids[k], "weight holds ", has ? weights[k]->numel() : 0,
                    " values for ", n_ids[k], " ids");
        parts.push_back(has ? weights[k]->reshape({-1}).to(opt) : at::ones({n_ids[k]}, opt));
      }
      weight = n == 1 ? parts[0].contiguous() : at::cat(parts);
      // (the backward of one weighted id per segment walks the segments like any other)
      if (unit_path) back_offsets = GroupOffsets(offsets, segments, widths, n_ids);
    }
    if (unit_path) {
      out = ExpandRows(plan, index, weight.defined() ? c10::optional<at::Tensor>(weight) : c10::nullopt, c10::nullopt,
                       c10::nullopt);
    } else {
      at::Tensor rev = plan->inverse(), table = block_ptr_table(chunks);
      out = at::empty({total_segments, D}, chunks[0].options());
      if (recorded && NotesOccurrences(plan->n(), total_segments, weight.defined()))
        occ = at::empty({plan->n()}, index.options());
      else if (recorded)
        plan->NotePool(merged, weight, mean);
      check(recis_segment_reduce_forward_blocks_occ(
          reinterpret_cast<const void* const*>(table.data_ptr()), static_cast<int64_t>(chunks.size()), emb->ChunkRows(),
          recis::hipabi::row_pitch_bytes(chunks[0]), index.data_ptr<int64_t>(), dtype_code(dtype_),
          weight.defined() ? weight.data_ptr() : nullptr, weight.defined() ? dtype_code(weight.scalar_type()) : 0,
          rev.data_ptr(), 0, merged.data_ptr(), index_kind(merged, "offsets"), out.data_ptr(), dtype_code(dtype_), plan->n(),
          index.numel(), total_segments, D, mean ? RECIS_MEAN : RECIS_SUM,
          occ.defined() ? occ.data_ptr() : nullptr, stream_of(device_)));
    }
    for (size_t k = 0; k < n; ++k) shapes[k] = {segments[k], D};
  }
  std::shared_ptr<LookupBackward> node;
  if (recorded) {
    node = std::make_shared<LookupBackward>();
    node->table = c10::intrusive_ptr<Hashtable>::reclaim_copy(this);
    node->plan = plan;
    node->saved_index = SavedVariable(index, false);
    node->saved_offsets = SavedVariable(back_offsets, false);
    node->saved_weight = SavedVariable(weight, false);
    node->occ = occ;
    node->mean = mean;
    node->tile = tile;
    node->split = split;
    node->first_shape = shapes[0];
    if (tile) {
      node->batch = segments;
      node->seq = tile_len;
    }
  }
  return std::make_tuple(outputs_of(out, shapes, split, node), plan,
                         merged.defined() ? TensorOrNone(merged) : TensorOrNone(c10::nullopt), index);
}

void Hashtable::AcceptTileGrad(const at::Tensor& index, const BatchPlanPtr& plan, const at::Tensor& offsets,
                               const std::vector<int64_t>& batch, const std::vector<int64_t>& seq,
                               const std::vector<at::Tensor>& grads) {
  const int64_t D = slot_group_->EmbSlot()->FlatSize();
  at::Tensor like;
  for (const auto& g : grads)
    if (g.defined() && !like.defined()) like = g;
  if (!like.defined()) return;  // no gradient reached any part
  at::Tensor src = plan->SrcForTile(batch, seq, offsets);
  std::vector<at::Tensor> parts;
  bool one_type = true;
  for (size_t k = 0; k < grads.size(); ++k) {
    const int64_t rows = batch[k] * seq[k];
    parts.push_back(grads[k].defined() ? grads[k].reshape({rows, D}) : at::zeros({rows, D}, like.options()));
    one_type = one_type && parts[k].scalar_type() == parts[0].scalar_type();
  }
  const bool apart = parts.size() <= 8 && one_type;
  std::vector<at::Tensor> rows = apart ? parts : std::vector<at::Tensor>{at::cat(parts)};
  AcceptPlannedGrad(SettledRows(index, plan), plan, rows, apart, src, c10::nullopt, c10::nullopt, plan->serial(), false);
}
