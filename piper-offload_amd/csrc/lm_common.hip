// lm_common.hip -- ABI version, error reporting, workspace sizing, factor prep.
#include "lm_impl.h"

static thread_local std::string g_err;

int lm_fail_v(int code, const char* fmt, va_list ap) {
  char buf[512];
  vsnprintf(buf, sizeof buf, fmt, ap);
  g_err = buf;
  return code;
}

extern "C" int lm_version(void) { return LM_ABI_VERSION; }
extern "C" const char* lm_last_error(void) { return g_err.c_str(); }
extern "C" size_t lm_workspace_size(int64_t M, int64_t N, int32_t rank) { return ws_layout(M, N, rank).total; }

// ---- kernel timer -----------------------------------------------------------
#include <atomic>
#include <map>
#include <mutex>
#include <vector>

namespace {
struct TimerRec {
  std::vector<std::pair<hipEvent_t, hipEvent_t>> pairs;
  hipEvent_t open = nullptr;
};
std::atomic<bool> g_timer_on{false};
std::mutex g_timer_mu;
std::map<std::string, TimerRec> g_timer;

void timer_clear_locked() {
  for (auto& kv : g_timer) {
    for (auto& p : kv.second.pairs) {
      (void)hipEventDestroy(p.first);
      (void)hipEventDestroy(p.second);
    }
    if (kv.second.open) (void)hipEventDestroy(kv.second.open);
  }
  g_timer.clear();
}
}  // namespace

bool lm_timer_on() { return g_timer_on.load(std::memory_order_relaxed); }

void lm_timer_mark(const char* family, hipStream_t st, bool begin) {
  std::lock_guard<std::mutex> lk(g_timer_mu);
  TimerRec& r = g_timer[family];
  hipEvent_t e;
  if (hipEventCreate(&e) != hipSuccess) return;
  (void)hipEventRecord(e, st);
  if (begin) {
    if (r.open) (void)hipEventDestroy(r.open);
    r.open = e;
  } else if (r.open) {
    r.pairs.emplace_back(r.open, e);
    r.open = nullptr;
  } else {
    (void)hipEventDestroy(e);
  }
}

extern "C" int lm_timer_enable(int32_t enable) {
  std::lock_guard<std::mutex> lk(g_timer_mu);
  timer_clear_locked();
  g_timer_on.store(enable != 0);
  return LM_OK;
}

extern "C" int lm_timer_read(const char* family, double* total_ms, int64_t* launches) {
  std::lock_guard<std::mutex> lk(g_timer_mu);
  double ms = 0.0;
  int64_t n = 0;
  auto it = g_timer.find(family ? family : "");
  if (it != g_timer.end()) {
    for (auto& p : it->second.pairs) {
      HIP_TRY(hipEventSynchronize(p.second));
      float t = 0.0f;
      HIP_TRY(hipEventElapsedTime(&t, p.first, p.second));
      ms += t;
      ++n;
    }
  }
  if (total_ms) *total_ms = ms;
  if (launches) *launches = n;
  return LM_OK;
}

int launch_prep(const PrepItem& it, hipStream_t st) {
  TimedLaunch timed("prep", st);
  int64_t total = prep_units(it);
  int64_t blocks = (total + 255) / 256;
  if (blocks > 4096) blocks = 4096;
  hipLaunchKernelGGL(k_prep1, dim3((unsigned)blocks), dim3(256), 0, st, it, total);
  LAUNCH_CHECK();
  return LM_OK;
}


// ---- host -> device staging of descriptor tables ---------------------------
// The stack entries upload per-call descriptor tables.  Large ones go through a
// small pool of pinned host buffers, each guarded by an event recorded after
// its copy, so the entry points return without synchronizing the stream: a
// buffer is reused once its previous copy has completed (waiting on the
// oldest one when all are in flight).
namespace {
struct StageSlot {
  void* host = nullptr;
  size_t cap = 0;
  hipEvent_t ev = nullptr;
  int device = -1;
  uint64_t stamp = 0;
};
std::mutex g_stage_mu;
std::vector<StageSlot> g_stage;
uint64_t g_stage_clock = 0;
constexpr size_t kStageSlots = 8;
}  // namespace

// Small tables travel as kernel arguments (kUploadBytes per launch): a copy
// between two kernels of a stream, through whatever engine, costs about 15 us
// of idle GPU around its 4 us, a launch about 2 us and no staging slot.  Up to
// kUploadLaunches of them; a larger table is one copy.
namespace {
constexpr size_t kUploadBytes = 3584;  // kernel arguments end at 4 KiB
constexpr size_t kUploadLaunches = 4;
struct UploadChunk {
  uint32_t w[kUploadBytes / 4];
};
__global__ __launch_bounds__(256) void k_upload(UploadChunk c, uint32_t* dst, int words) {
  for (int i = threadIdx.x; i < words; i += 256) ((LM_GLOBAL uint32_t*)dst)[i] = c.w[i];
}
}  // namespace

// dst 4-byte aligned; whole words are written (the tables' regions are padded)
static int upload_args(uint8_t* dst, const uint8_t* src, size_t bytes, hipStream_t st) {
  for (size_t off = 0; off < bytes; off += kUploadBytes) {
    const size_t n = bytes - off < kUploadBytes ? bytes - off : kUploadBytes;
    UploadChunk c;
    memcpy(c.w, src + off, n);
    if (n % 4) memset((uint8_t*)c.w + n, 0, 4 - n % 4);
    hipLaunchKernelGGL(k_upload, dim3(1), dim3(256), 0, st, c, (uint32_t*)(dst + off), (int)((n + 3) / 4));
    LAUNCH_CHECK();
  }
  return LM_OK;
}

int lm_stage_h2d(void* dst, const void* src, size_t bytes, hipStream_t st) {
  if (bytes == 0) return LM_OK;
  if (bytes <= kUploadBytes * kUploadLaunches) return upload_args((uint8_t*)dst, (const uint8_t*)src, bytes, st);
  int dev = 0;
  HIP_TRY(hipGetDevice(&dev));
  std::lock_guard<std::mutex> lk(g_stage_mu);
  StageSlot* pick = nullptr;
  for (auto& s : g_stage)  // a free slot of this device that is large enough
    if (s.device == dev && s.cap >= bytes && hipEventQuery(s.ev) == hipSuccess) { pick = &s; break; }
  if (!pick && g_stage.size() < kStageSlots) {
    g_stage.emplace_back();
    pick = &g_stage.back();
    pick->device = dev;
    HIP_TRY(hipEventCreateWithFlags(&pick->ev, hipEventDisableTiming));
  }
  if (!pick) {  // every slot busy or too small: wait for the oldest of this device
    for (auto& s : g_stage)
      if (s.device == dev && (!pick || s.stamp < pick->stamp)) pick = &s;
    if (!pick) return fail(LM_EHIP, "no staging slot for device %d", dev);
    HIP_TRY(hipEventSynchronize(pick->ev));
  }
  if (pick->cap < bytes) {
    if (pick->host) HIP_TRY(hipHostFree(pick->host));
    pick->host = nullptr;
    pick->cap = 0;
    const size_t cap = bytes < 65536 ? 65536 : bytes * 2;
    HIP_TRY(hipHostMalloc(&pick->host, cap, hipHostMallocDefault));
    pick->cap = cap;
  }
  memcpy(pick->host, src, bytes);
  HIP_TRY(hipMemcpyAsync(dst, pick->host, bytes, hipMemcpyHostToDevice, st));
  HIP_TRY(hipEventRecord(pick->ev, st));
  pick->stamp = ++g_stage_clock;
  return LM_OK;
}
