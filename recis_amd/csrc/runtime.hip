// Host-side runtime shared by all entry points: thread-local error text, the
// per-device soft-error word, and per-(device, stream) scratch memory.
#include <stdarg.h>
#include <stdio.h>

#include <atomic>
#include <map>
#include <mutex>
#include <string>
#include <utility>
#include <vector>

#include "common.cuh"

namespace recis_hip {

static thread_local char g_err[512] = "";

void set_error(const char* fmt, ...) {
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(g_err, sizeof(g_err), fmt, ap);
  va_end(ap);
}

int fail(int code, const char* fmt, ...) {
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(g_err, sizeof(g_err), fmt, ap);
  va_end(ap);
  return code;
}

int current_device() {
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess) return -1;
  return dev;
}

static std::mutex g_mu;

// The soft-error word lives in the code object of this library (one copy per device that loads
// it), so reaching it never allocates: entry points that must not allocate can use it too.
static __device__ int g_error_word[4];
constexpr int kMaxDevices = 64;
static int* g_err_words[kMaxDevices];

int* device_error_word(int device) {
  if (device < 0 || device >= kMaxDevices) return nullptr;
  std::lock_guard<std::mutex> l(g_mu);
  if (g_err_words[device]) return g_err_words[device];
  int cur = -1;
  if (hipGetDevice(&cur) != hipSuccess) return nullptr;
  if (cur != device && hipSetDevice(device) != hipSuccess) return nullptr;
  void* p = nullptr;
  const hipError_t rc = hipGetSymbolAddress(&p, HIP_SYMBOL(g_error_word));
  if (cur != device) (void)hipSetDevice(cur);
  if (rc != hipSuccess) return nullptr;
  g_err_words[device] = static_cast<int*>(p);
  return g_err_words[device];
}

// A pinned word per device: not zero once a kernel that looks has found bits in the error word. The host reads it
// without waiting, for calls that have no count to come with the bits.
static std::atomic<int*> g_report_words[kMaxDevices];

int* error_report_word(int device) {
  if (device < 0 || device >= kMaxDevices) return nullptr;
  if (int* known = g_report_words[device].load(std::memory_order_acquire)) return known;
  std::lock_guard<std::mutex> l(g_mu);
  if (int* known = g_report_words[device].load(std::memory_order_relaxed)) return known;
  void* p = nullptr;
  if (hipHostMalloc(&p, 64, hipHostMallocPortable) != hipSuccess) return nullptr;
  *static_cast<volatile int*>(p) = 0;
  g_report_words[device].store(static_cast<int*>(p), std::memory_order_release);
  return static_cast<int*>(p);
}

struct Workspace {
  void* ptr = nullptr;
  size_t bytes = 0;
};
static std::map<std::pair<int, hipStream_t>, Workspace> g_ws;

int get_workspace(hipStream_t stream, size_t bytes, void** out) {
  int dev = current_device();
  std::lock_guard<std::mutex> l(g_mu);
  Workspace& w = g_ws[std::make_pair(dev, stream)];
  if (w.bytes < bytes) {
    // Work already queued on this stream may still read the old buffer:
    // drain the stream before the buffer is replaced.
    if (w.ptr) {
      RECIS_CHECK_HIP(hipStreamSynchronize(stream));
      RECIS_CHECK_HIP(hipFree(w.ptr));
      w.ptr = nullptr;
      w.bytes = 0;
    }
    size_t want = bytes < (size_t(1) << 20) ? (size_t(1) << 20) : bytes + bytes / 4;
    want = (want + 255) & ~size_t(255);
    RECIS_CHECK_HIP(hipMalloc(&w.ptr, want));
    w.bytes = want;
  }
  *out = w.ptr;
  return RECIS_OK;
}

// Pinned words and an event for the count of a plan. A slot belongs to one (device, stream), so that whoever takes it
// next writes behind the kernels of whoever had it before. It is held by the thread that staged a count with it, until that
// thread stages another; or by a ticket, until the ticket is given back: never handed out while a count in it may still be read.
struct CountSlot {
  int64_t* host = nullptr;
  hipEvent_t event = nullptr;
  int dev = -1;
  hipStream_t stream = nullptr;
  const void* holder = nullptr;  // the thread (its t_staged), NULL with a ticket or when free
  int64_t ticket = -1;
};
struct CountStaging {
  std::vector<CountSlot*> free;
  CountSlot* last = nullptr;     // the stream's last staged count
  int64_t* flag_word = nullptr;  // pinned, see get_flag_word
};
constexpr int kSlotChunk = 32;      // slots of one pinned allocation
constexpr size_t kMaxTickets = 4096;  // outstanding at once (a plan without one reads its own device word)
// (never destroyed: threads and plans may outlive this library's static objects)
static auto& g_staging = *new std::map<std::pair<int, hipStream_t>, CountStaging>;
static auto& g_tickets = *new std::map<int64_t, CountSlot*>;
static int64_t g_next_ticket = 1;

struct StagedHere {  // the last count this thread staged
  CountSlot* slot = nullptr;
  ~StagedHere();
};
static thread_local StagedHere t_staged;

static void give_back_held() {  // g_mu is held
  CountSlot* s = t_staged.slot;
  t_staged.slot = nullptr;
  if (s == nullptr || s->holder != &t_staged) return;
  s->holder = nullptr;
  g_staging[std::make_pair(s->dev, s->stream)].free.push_back(s);
}
StagedHere::~StagedHere() {
  std::lock_guard<std::mutex> l(g_mu);
  give_back_held();
}

int get_count_staging(hipStream_t stream, int64_t** host, hipEvent_t* event) {
  const int dev = current_device();
  std::lock_guard<std::mutex> l(g_mu);
  give_back_held();
  CountStaging& c = g_staging[std::make_pair(dev, stream)];
  if (c.free.empty()) {
    int64_t* words = nullptr;
    RECIS_CHECK_HIP(hipHostMalloc(reinterpret_cast<void**>(&words), 64 * kSlotChunk, hipHostMallocDefault));
    for (int w = 0; w < 8 * kSlotChunk; ++w) words[w] = 0;
    for (int k = kSlotChunk - 1; k >= 0; --k) {
      CountSlot* s = new CountSlot;
      s->host = words + 8 * k;
      s->dev = dev;
      s->stream = stream;
      c.free.push_back(s);
    }
  }
  CountSlot* s = c.free.back();
  if (s->event == nullptr) RECIS_CHECK_HIP(hipEventCreateWithFlags(&s->event, hipEventDisableTiming));
  c.free.pop_back();
  s->holder = &t_staged;
  t_staged.slot = s;
  c.last = s;
  *host = s->host;
  *event = s->event;
  return RECIS_OK;
}

int get_flag_word(hipStream_t stream, int64_t** host) {
  const int dev = current_device();
  std::lock_guard<std::mutex> l(g_mu);
  CountStaging& c = g_staging[std::make_pair(dev, stream)];
  if (c.flag_word == nullptr)
    RECIS_CHECK_HIP(hipHostMalloc(reinterpret_cast<void**>(&c.flag_word), 64, hipHostMallocDefault));
  *host = c.flag_word;
  return RECIS_OK;
}

bool last_count_staging(hipStream_t stream, int64_t** host, hipEvent_t* event) {
  const int dev = current_device();
  std::lock_guard<std::mutex> l(g_mu);
  CountSlot* s = t_staged.slot;
  if (s == nullptr || s->dev != dev || s->stream != stream) s = g_staging[std::make_pair(dev, stream)].last;
  if (s == nullptr) return false;
  *host = s->host;
  *event = s->event;
  return true;
}

int64_t take_count_ticket(hipStream_t stream) {
  const int dev = current_device();
  std::lock_guard<std::mutex> l(g_mu);
  CountSlot* s = t_staged.slot;
  if (s == nullptr || s->dev != dev || s->stream != stream) return -1;
  if (s->holder == &t_staged && g_tickets.size() < kMaxTickets) {
    s->holder = nullptr;
    s->ticket = g_next_ticket++;
    g_tickets[s->ticket] = s;
    t_staged.slot = nullptr;
    return s->ticket;
  }
  return -1;
}

bool find_count_ticket(int64_t ticket, int64_t** host, hipEvent_t* event) {
  std::lock_guard<std::mutex> l(g_mu);
  auto it = g_tickets.find(ticket);
  if (it == g_tickets.end()) return false;
  *host = it->second->host;
  *event = it->second->event;
  return true;
}

void give_count_ticket(int64_t ticket) {
  std::lock_guard<std::mutex> l(g_mu);
  auto it = g_tickets.find(ticket);
  if (it == g_tickets.end()) return;
  CountSlot* s = it->second;
  g_tickets.erase(it);
  s->ticket = -1;
  g_staging[std::make_pair(s->dev, s->stream)].free.push_back(s);
}

bool g_profile_on = false;

struct TimedLaunch {
  const char* name;
  hipEvent_t start, stop;
};
static std::vector<TimedLaunch> g_timed;

void KernelTimer::begin(const char* name, hipStream_t stream) {
  std::lock_guard<std::mutex> l(g_mu);
  TimedLaunch t;
  t.name = name;
  if (hipEventCreate(&t.start) != hipSuccess || hipEventCreate(&t.stop) != hipSuccess) {
    active_ = false;
    return;
  }
  (void)hipEventRecord(t.start, stream);
  g_timed.push_back(t);
  slot_ = static_cast<int>(g_timed.size()) - 1;
  stream_ = stream;
}

void KernelTimer::end() {
  std::lock_guard<std::mutex> l(g_mu);
  if (slot_ >= 0 && slot_ < static_cast<int>(g_timed.size())) (void)hipEventRecord(g_timed[slot_].stop, stream_);
}

}  // namespace recis_hip

extern "C" {

int recis_hip_profile_enable(int on) {
  std::lock_guard<std::mutex> l(recis_hip::g_mu);
  recis_hip::g_profile_on = on != 0;
  return RECIS_OK;
}

int recis_hip_profile_report(char* buf, int64_t cap) {
  using namespace recis_hip;
  RECIS_REQUIRE(buf != nullptr && cap > 0, "buf must hold the report");
  RECIS_CHECK_HIP(hipDeviceSynchronize());
  std::lock_guard<std::mutex> l(g_mu);
  std::map<std::string, std::pair<int64_t, double>> agg;
  for (auto& t : g_timed) {
    float ms = 0.f;
    if (hipEventElapsedTime(&ms, t.start, t.stop) == hipSuccess) {
      auto& a = agg[t.name];
      a.first += 1;
      a.second += ms;
    }
    (void)hipEventDestroy(t.start);
    (void)hipEventDestroy(t.stop);
  }
  g_timed.clear();
  std::string out;
  char line[256];
  for (auto& kv : agg) {
    snprintf(line, sizeof(line), "%s %lld %.6f\n", kv.first.c_str(), (long long)kv.second.first, kv.second.second);
    out += line;
  }
  snprintf(buf, static_cast<size_t>(cap), "%s", out.c_str());
  return RECIS_OK;
}

const char* recis_hip_last_error(void) { return recis_hip::g_err; }

int recis_hip_abi_version(void) { return RECIS_HIP_ABI_VERSION; }

int recis_hip_poll_device_errors(int* bits) {
  using namespace recis_hip;
  RECIS_REQUIRE(bits != nullptr, "bits must not be NULL");
  int dev = current_device();
  int* w = device_error_word(dev);
  RECIS_REQUIRE(w != nullptr, "could not reach the device error word");
  RECIS_CHECK_HIP(hipDeviceSynchronize());
  if (int* reported = error_report_word(dev)) *static_cast<volatile int*>(reported) = 0;
  RECIS_CHECK_HIP(hipMemcpy(bits, w, sizeof(int), hipMemcpyDeviceToHost));
  if (*bits) RECIS_CHECK_HIP(hipMemset(w, 0, sizeof(int)));
  return RECIS_OK;
}

int recis_hip_device_errors_reported(int* reported) {
  using namespace recis_hip;
  RECIS_REQUIRE(reported != nullptr, "reported must not be NULL");
  const int* w = error_report_word(current_device());
  RECIS_REQUIRE(w != nullptr, "could not reach the error report word");
  *reported = *static_cast<const volatile int*>(w);
  return RECIS_OK;
}

}  // extern "C"
