// hoststage.cpp -- see hoststage.hpp.
//
// A copy to pageable memory runs at 16-18 GB/s here (3.2 MB: 185 us, 64 MB: 3.6 ms, and as
// much again for the first touch of a fresh array), one to pinned memory at 50-57 GB/s.  The
// chunks of a download go to the two halves of a pinned buffer in turn, and while one is in
// flight the threads of the host copy the other into the caller's memory, first touch and all
// (3.2 MB: 268 -> 176 us with the output pass, 64 MB into fresh arrays: 6.1 -> 2.8 ms).
#include "hoststage.hpp"

#include <omp.h>

#include <algorithm>
#include <atomic>
#include <cstring>
#include <mutex>

#include "devbuf.hpp"

namespace fmmh {

namespace {

constexpr size_t kHalf = size_t(4) << 20;   // bytes per half
constexpr size_t kSlice = size_t(128) << 10;  // bytes per host thread at least
constexpr int kThreads = 16;
constexpr int kTeams = 4;                   // calling threads with copying threads of their own
constexpr size_t kKeep = 8;                 // idle buffers kept (one for each GPU of a node)

struct Stage {
  int device = 0;
  char *buf = nullptr;
  hipEvent_t done[2] = {nullptr, nullptr};
};

std::mutex g_mu;
std::vector<Stage> g_idle;
int g_users = 0;

void destroy(Stage &t) {
  for (hipEvent_t e : t.done)
    if (e) (void)hipEventDestroy(e);
  if (t.buf) (void)hipHostFree(t.buf);
}

// An idle buffer of the device, or a new one (the calling thread's current device must be it:
// the events belong to that one); false when none can be had.
bool take(int device, Stage &t) {
  {
    std::lock_guard<std::mutex> lock(g_mu);
    for (size_t i = 0; i < g_idle.size(); ++i)
      if (g_idle[i].device == device) {
        t = g_idle[i];
        g_idle.erase(g_idle.begin() + long(i));
        return true;
      }
  }
  t = Stage{};
  t.device = device;
  void *p = nullptr;
  bool ok = hipHostMalloc(&p, 2 * kHalf, hipHostMallocDefault) == hipSuccess;
  t.buf = static_cast<char *>(p);
  for (int k = 0; ok && k < 2; ++k) ok = hipEventCreateWithFlags(&t.done[k], hipEventDisableTiming) == hipSuccess;
  if (!ok) {
    destroy(t);
    (void)hipGetLastError();
  }
  return ok;
}

void give(Stage &t) {
  {
    std::lock_guard<std::mutex> lock(g_mu);
    if (g_users > 0 && g_idle.size() < kKeep) {
      g_idle.push_back(t);
      return;
    }
  }
  destroy(t);
}

// The thread's current device is `device` while this lives.
class OnDevice {
 public:
  explicit OnDevice(int device) {
    hip_check(hipGetDevice(&before_), "hipGetDevice");
    if (before_ != device) hip_check(hipSetDevice(device), "hipSetDevice");
    moved_ = before_ != device;
  }
  ~OnDevice() {
    if (moved_) (void)hipSetDevice(before_);
  }

 private:
  int before_ = 0;
  bool moved_ = false;
};

// Whether the runtime knows this memory (pinned, managed or a GPU's): it copies there itself.
bool known(const void *p) {
  hipPointerAttribute_t a{};
  if (hipPointerGetAttributes(&a, p) != hipSuccess) {
    (void)hipGetLastError();
    return false;
  }
  return a.type != hipMemoryTypeUnregistered;
}

// An OpenMP team belongs to the thread that opened it and stays as long as that one, so only a few
// threads at a time may have one, the others copy alone.  (One set of threads for the process,
// woken through a condition variable: 100,000 points' outputs 163 -> 402 us, since a team
// still spins when the next chunk comes.)
class Team {
 public:
  Team() = default;
  ~Team() {
    if (mine_) --count_;
  }
  bool have() {
    if (!mine_ && !(mine_ = count_.fetch_add(1) < kTeams)) --count_;
    return mine_;
  }

 private:
  static std::atomic<int> count_;
  bool mine_ = false;
};
std::atomic<int> Team::count_{0};
thread_local Team t_team;

void host_copy(char *dst, const char *src, size_t bytes) {
  const int n = int(std::min<size_t>(size_t(std::min(kThreads, omp_get_max_threads())), bytes / kSlice));
  if (n <= 1 || !t_team.have()) {
    std::memcpy(dst, src, bytes);
    return;
  }
  const size_t each = (bytes / size_t(n) + 4095) / 4096 * 4096;
#pragma omp parallel for num_threads(n) schedule(static, 1)
  for (int k = 0; k < n; ++k) {
    const size_t a = std::min(bytes, size_t(k) * each), b = k + 1 == n ? bytes : std::min(bytes, a + each);
    if (b > a) std::memcpy(dst + a, src + a, b - a);
  }
}

}  // namespace

HostStageUser::HostStageUser() {
  std::lock_guard<std::mutex> lock(g_mu);
  g_idle.reserve(kKeep);  // giving a buffer back cannot fail
  ++g_users;
}

HostStageUser::~HostStageUser() {
  std::vector<Stage> gone;
  {
    std::lock_guard<std::mutex> lock(g_mu);
    if (--g_users == 0) gone.swap(g_idle);
  }
  for (Stage &t : gone) destroy(t);
}

void HostStageUser::download(int device, hipStream_t s, const std::vector<HostCopy> &copies) {
  size_t total = 0;
  for (const HostCopy &c : copies) total += c.bytes;
  if (total == 0) return;
  const OnDevice on(device);
  // chunks of a quarter of the whole, so that copying starts early, within the halves' size
  const size_t most = std::min(kHalf, std::max<size_t>(size_t(256) << 10, (total / 4 + 4095) / 4096 * 4096));
  std::vector<HostCopy> chunks;
  for (const HostCopy &c : copies)
    for (size_t at = 0; at < c.bytes; at += most)
      chunks.push_back({static_cast<char *>(c.dst) + at, static_cast<const char *>(c.src) + at,
                        std::min(most, c.bytes - at)});
  // A few kilobytes arrive sooner through the runtime's own staging, and pinned memory sooner
  // without one (4M points' outputs, 128 MB: 2.5 ms against 3.1).
  bool direct = total < (size_t(64) << 10);
  for (const HostCopy &c : copies) direct = direct || (c.bytes && known(c.dst));
  Stage t;
  if (direct || !take(device, t)) {
    for (const HostCopy &c : copies)
      if (c.bytes) hip_check(hipMemcpyAsync(c.dst, c.src, c.bytes, hipMemcpyDeviceToHost, s), "download");
    hip_check(hipStreamSynchronize(s), "download");
    return;
  }
  const auto send = [&](size_t i) {
    const HostCopy &c = chunks[i];
    const hipError_t e = hipMemcpyAsync(t.buf + (i & 1) * kHalf, c.src, c.bytes, hipMemcpyDeviceToHost, s);
    return e != hipSuccess ? e : hipEventRecord(t.done[i & 1], s);
  };
  hipError_t err = send(0);
  for (size_t i = 0; err == hipSuccess && i < chunks.size(); ++i) {
    if (i + 1 < chunks.size()) err = send(i + 1);
    if (err == hipSuccess) err = hipEventSynchronize(t.done[i & 1]);
    if (err == hipSuccess) host_copy(static_cast<char *>(chunks[i].dst), t.buf + (i & 1) * kHalf, chunks[i].bytes);
  }
  if (err != hipSuccess) {
    // the stream may still write the buffer: wait before it is freed
    (void)hipStreamSynchronize(s);
    destroy(t);
    hip_check(err, "download");
  }
  give(t);
}

}  // namespace fmmh
