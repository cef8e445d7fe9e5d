#include "plan.h"

#include <atomic>

#include "abi_util.h"
#include "ops.h"

namespace recis {

using namespace recis::hipabi;

namespace {

constexpr int64_t kPlanJobs = 64;  // arrays one recis_unique_plan_jobs call takes

std::atomic<int64_t> g_serial{1};

std::string describe_device_errors(int bits) {
  std::string s;
  auto add = [&](int bit, const char* text) {
    if (bits & bit) {
      if (!s.empty()) s += "; ";
      s += text;
    }
  };
  add(RECIS_DEVERR_INDEX_RANGE, "an index outside the rows / blocks the caller passed");
  add(RECIS_DEVERR_OFFSETS, "offsets not monotone or out of range");
  add(RECIS_DEVERR_TABLE_FULL, "the id map found no free slot");
  add(RECIS_DEVERR_PLAN_OVERFLOW, "batch plan: too many distinct ids in one hash bucket");
  return s + " (bits " + std::to_string(bits) + ")";
}

at::Tensor flat_ids(const at::Tensor& t) {
  require_gpu(t, "ids");
  if (t.dim() == 1 && t.scalar_type() == at::kLong && t.is_contiguous()) return t;
  return t.to(at::kLong).contiguous().view({-1});
}

// The bits that travelled to the host with a staged count (-1: not known) as an exception.
void raise_device_errors(int bits) {
  if (bits == 0) return;
  int polled = 0;
  check(recis_hip_poll_device_errors(&polled));  // waits for the device and clears the word
  // (two counts that were under way together carry one error's bits twice: it is raised once)
  TORCH_CHECK(polled == 0, "librecis_hip: device-side errors in earlier kernels: ", describe_device_errors(polled));
}

}  // namespace

void raise_reported_errors() {
  int reported = 0;
  check(recis_hip_device_errors_reported(&reported));
  if (reported) raise_device_errors(-1);
}

BatchPlanPtr BatchPlan::Make(const std::vector<at::Tensor>& ids_in, const c10::optional<std::vector<int64_t>>& tags,
                             recis_idmap* map, bool wait, bool need_inverse, bool need_pos) {
  TORCH_CHECK(!tags.has_value() || tags->size() == ids_in.size(), "unique_plan: ", tags.has_value() ? tags->size() : 0,
              " tags for ", ids_in.size(), " id tensors");
  std::vector<at::Tensor> jobs;
  jobs.reserve(ids_in.size());
  for (const auto& t : ids_in) jobs.push_back(flat_ids(t));
  if (jobs.empty() || static_cast<int64_t>(jobs.size()) > kPlanJobs) {
    // too many arrays for one call (or none): make the batch first
    TORCH_CHECK(!jobs.empty(), "unique_plan: no id tensors");
    at::Tensor batch;
    if (tags.has_value()) {
      batch = functional::ids_encode(jobs, at::tensor(*tags, at::TensorOptions().dtype(at::kLong)));
    } else {
      batch = at::cat(jobs);
    }
    jobs.assign(1, batch);
  }
  const bool tagged = tags.has_value() && ids_in.size() == jobs.size();
  int64_t n = 0;
  for (const auto& t : jobs) n += t.numel();
  const at::Device dev = jobs[0].device();
  c10::DeviceGuard guard(dev);
  auto p = c10::make_intrusive<BatchPlan>();
  p->serial_ = g_serial.fetch_add(1);
  p->n_ = n;
  auto i64 = at::TensorOptions().device(dev).dtype(at::kLong);
  auto i32 = at::TensorOptions().device(dev).dtype(at::kInt);
  p->unique_buf_ = at::empty({n}, i64);
  if (need_inverse) p->inverse_ = at::empty({n}, i32);
  p->row_start_ = at::empty({n + 1}, i32);
  p->occ_ = at::empty({n}, i32);
  if (need_pos) p->pos_ = at::empty({n}, i32);
  p->hot_cap_ = n / RECIS_PLAN_HOT_LEN + n / RECIS_PLAN_HOT_CHUNK + 2;
  p->hot_items_ = at::empty({2 * p->hot_cap_}, i32);
  p->counts_ = at::empty({2}, i64);
  if (map != nullptr) p->index_buf_ = at::empty({n}, i64);
  p->stream_ = stream_of(dev);
  int64_t count = 0;
  auto ptrs = host_ptrs<int64_t>(jobs);
  auto sizes = numels(jobs);
  auto i32p = [](const at::Tensor& t) { return t.defined() ? t.data_ptr<int32_t>() : nullptr; };
  check(recis_unique_plan_jobs(map, ptrs.data(), sizes.data(), tagged ? tags->data() : nullptr,
                               static_cast<int64_t>(jobs.size()), p->unique_buf_.data_ptr<int64_t>(), i32p(p->inverse_),
                               i32p(p->row_start_), i32p(p->occ_), i32p(p->pos_), i32p(p->hot_items_), p->hot_cap_,
                               p->counts_.data_ptr<int64_t>(),
                               p->index_buf_.defined() ? p->index_buf_.data_ptr<int64_t>() : nullptr,
                               wait ? &count : nullptr, wait ? 0 : RECIS_PLAN_STAGE_COUNT, p->stream_));
  check(recis_unique_plan_ticket(&p->ticket_, p->stream_));
  if (wait) p->U();
  return p;
}

int64_t BatchPlan::U() {
  if (U_ >= 0) return U_;
  c10::DeviceGuard guard(device());
  int64_t count = -1;
  int bits = 0;
  check(recis_unique_plan_count_of(ticket_, 1, &count, &bits, stream_));
  if (count < 0) {  // no ticket was left for this plan: its own device words
    count = counts_[0].item<int64_t>();
    bits = -1;
  }
  U_ = count;
  GiveTicket();
  raise_device_errors(bits);
  return U_;
}

void BatchPlan::GiveTicket() {
  if (ticket_ >= 0) recis_unique_plan_release(ticket_);
  ticket_ = -1;
}

at::Tensor BatchPlan::unique() {
  if (!unique_.defined()) unique_ = unique_buf_.narrow(0, 0, U());
  return unique_;
}

void BatchPlan::FillLate() {
  c10::DeviceGuard guard(device());
  auto i32 = at::TensorOptions().device(device()).dtype(at::kInt);
  at::Tensor inv = inverse_.defined() ? at::Tensor() : at::empty({n_}, i32);
  at::Tensor pos = pos_.defined() ? at::Tensor() : at::empty({n_}, i32);
  if (n_) {
    check(recis_plan_inverse_from_lists(row_start_.data_ptr<int32_t>(), occ_.data_ptr<int32_t>(),
                                        counts_.data_ptr<int64_t>(), n_, inv.defined() ? inv.data_ptr<int32_t>() : nullptr,
                                        pos.defined() ? pos.data_ptr<int32_t>() : nullptr, stream_of(device())));
  }
  if (inv.defined()) inverse_ = inv;
  if (pos.defined()) pos_ = pos;
}

at::Tensor BatchPlan::inverse() {
  if (!inverse_.defined()) FillLate();
  return inverse_;
}

at::Tensor BatchPlan::pos() {
  if (!pos_.defined()) FillLate();
  return pos_;
}

int64_t BatchPlan::LookupCall(const void* owner) const {
  for (auto it = lookup_calls_.rbegin(); it != lookup_calls_.rend(); ++it) {
    if (it->first == owner) return it->second;
  }
  return 0;
}

std::tuple<at::Tensor, at::Tensor, at::Tensor> BatchPlan::FillLists(const at::Tensor& offsets_in,
                                                                    const at::Tensor& weight_in, bool mean,
                                                                    bool want_pool, const std::vector<int64_t>* batch,
                                                                    const std::vector<int64_t>* seq) {
  require_gpu(offsets_in, "offsets");
  at::Tensor offsets = offsets_in.contiguous();
  const at::Device dev = offsets.device();
  c10::DeviceGuard guard(dev);
  const int64_t S = offsets.numel() - 1;
  auto i32 = at::TensorOptions().device(dev).dtype(at::kInt);
  at::Tensor src, coef, tile, weight;
  if (weight_in.defined()) {
    require_gpu(weight_in, "weight");
    weight = weight_in.contiguous();
  }
  if (want_pool) {
    src = at::empty({n_}, i32);
    if (weight.defined() || mean) coef = at::empty({n_}, i32.dtype(at::kFloat));
  }
  if (batch != nullptr) {
    TORCH_CHECK(batch->size() == seq->size(), "batch and seq differ in length");
    tile = at::empty({n_}, i32);
  }
  if (n_) {
    check(recis_csr_fill_lists(occ_.data_ptr<int32_t>(), n_, offsets.data_ptr(), index_kind(offsets, "offsets"), S,
                               weight.defined() ? weight.data_ptr() : nullptr,
                               weight.defined() ? dtype_code(weight.scalar_type()) : 0, mean ? 1 : 0,
                               src.defined() ? src.data_ptr<int32_t>() : nullptr,
                               coef.defined() ? coef.data_ptr<float>() : nullptr, batch ? batch->data() : nullptr,
                               batch ? seq->data() : nullptr, batch ? static_cast<int64_t>(batch->size()) : 0,
                               tile.defined() ? tile.data_ptr<int32_t>() : nullptr, stream_of(dev)));
  }
  return std::make_tuple(src, coef, tile);
}

std::tuple<at::Tensor, c10::optional<at::Tensor>> BatchPlan::SrcCoefForPool(const at::Tensor& offsets,
                                                                             const c10::optional<at::Tensor>& weight,
                                                                             bool mean) {
  const bool has_w = weight.has_value() && weight->defined();
  const void* wp = has_w ? weight->data_ptr() : nullptr;
  if (fill_valid_ && fill_offsets_ == offsets.data_ptr() && fill_weight_ == wp && fill_mean_ == mean) {
    return std::make_tuple(fill_src_, fill_coef_.defined() ? c10::optional<at::Tensor>(fill_coef_) : c10::nullopt);
  }
  auto filled = FillLists(offsets, has_w ? *weight : at::Tensor(), mean, true, nullptr, nullptr);
  KeepPoolLists(offsets, has_w ? *weight : at::Tensor(), mean, std::get<0>(filled), std::get<1>(filled));
  return std::make_tuple(fill_src_, fill_coef_.defined() ? c10::optional<at::Tensor>(fill_coef_) : c10::nullopt);
}

void BatchPlan::KeepPoolLists(const at::Tensor& offsets, const at::Tensor& weight, bool mean, const at::Tensor& src,
                              const at::Tensor& coef) {
  fill_offsets_ = offsets.data_ptr();
  fill_weight_ = weight.defined() ? weight.data_ptr() : nullptr;
  fill_keep_offsets_ = offsets;  // alive as long as the cache entry: its address cannot be handed out again
  fill_keep_weight_ = weight;
  fill_mean_ = mean;
  fill_valid_ = true;
  fill_src_ = src;
  fill_coef_ = coef;
}

void BatchPlan::NotePool(const at::Tensor& offsets, const at::Tensor& weight, bool mean) {
  note_offsets_ = offsets;
  note_weight_ = weight;
  note_mean_ = mean;
}

std::tuple<at::Tensor, c10::optional<at::Tensor>> BatchPlan::SrcCoefFromOcc(const at::Tensor& occ,
                                                                             const at::Tensor& offsets, bool coef) {
  c10::DeviceGuard guard(device());
  auto i32 = at::TensorOptions().device(device()).dtype(at::kInt);
  at::Tensor src = at::empty({n_}, i32), c;
  if (coef) c = at::empty({n_}, i32.dtype(at::kFloat));
  check(recis_csr_lists_from_occ(occ_.data_ptr<int32_t>(), n_, occ.data_ptr(), offsets.data_ptr(),
                                 index_kind(offsets, "offsets"), offsets.numel() - 1, src.data_ptr<int32_t>(),
                                 coef ? c.data_ptr<float>() : nullptr, stream_of(device())));
  return std::make_tuple(src, coef ? c10::optional<at::Tensor>(c) : c10::nullopt);
}

at::Tensor BatchPlan::SrcForTile(const std::vector<int64_t>& batch, const std::vector<int64_t>& seq,
                                 const at::Tensor& offsets) {
  if (note_offsets_.defined() && !fill_valid_ && note_offsets_.is_same(offsets)) {
    auto both = FillLists(offsets, note_weight_, note_mean_, true, &batch, &seq);
    KeepPoolLists(offsets, note_weight_, note_mean_, std::get<0>(both), std::get<1>(both));
    return std::get<2>(both);
  }
  return std::get<2>(FillLists(offsets, at::Tensor(), false, false, &batch, &seq));
}

std::tuple<at::Tensor, c10::optional<at::Tensor>, at::Tensor> BatchPlan::SrcForPoolAndTile(
    const at::Tensor& offsets, const c10::optional<at::Tensor>& weight, bool mean, const std::vector<int64_t>& batch,
    const std::vector<int64_t>& seq) {
  const at::Tensor w = weight.has_value() ? *weight : at::Tensor();
  auto filled = FillLists(offsets, w, mean, true, &batch, &seq);
  KeepPoolLists(offsets, w, mean, std::get<0>(filled), std::get<1>(filled));
  return std::make_tuple(fill_src_, fill_coef_.defined() ? c10::optional<at::Tensor>(fill_coef_) : c10::nullopt,
                         std::get<2>(filled));
}

BatchPlanPtr unique_plan(std::vector<at::Tensor> ids, c10::optional<std::vector<int64_t>> tags, int64_t idmap_handle,
                         bool wait, bool need_inverse, bool need_pos) {
  return BatchPlan::Make(ids, tags, reinterpret_cast<recis_idmap*>(idmap_handle), wait, need_inverse, need_pos);
}

}  // namespace recis
