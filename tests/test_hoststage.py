"""Downloads through pinned staging (fmm_amd/csrc/hoststage.cpp) on the host, over a stand-in for
the HIP runtime: two devices, events and streams bound to theirs, memory that is counted.  The
runtime's rule that an event is recorded on a stream of its own device needs more than one GPU
to be met, and the stand-in enforces it."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

RUNTIME = r"""
#include <hip/hip_runtime.h>
#include <atomic>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <stdexcept>
#include <thread>
#include <vector>
#include "hoststage.hpp"

namespace fmmh {
void hip_check(hipError_t e, const char *what) {
  if (e != hipSuccess) throw std::runtime_error(std::string(what) + " " + std::to_string(int(e)));
}
}  // namespace fmmh

static thread_local int g_device = 0;
static std::atomic<const void *> g_pinned{nullptr};
static std::atomic<bool> g_refuse_unknown{false};
static std::atomic<int> g_direct{0};
static std::atomic<int> g_buffers{0}, g_events{0}, g_fail_after{1 << 30};
struct Event { int device; };

static hipStream_t stream_of(int device) { return reinterpret_cast<hipStream_t>(uintptr_t(0x1000 + device)); }
static int device_of(hipStream_t s) { return int(reinterpret_cast<uintptr_t>(s)) - 0x1000; }

extern "C" {
hipError_t hipGetDevice(int *d) { *d = g_device; return hipSuccess; }
hipError_t hipSetDevice(int d) { g_device = d; return hipSuccess; }
hipError_t hipHostMalloc(void **p, size_t n, unsigned) { *p = std::malloc(n); ++g_buffers; return hipSuccess; }
hipError_t hipHostFree(void *p) { std::free(p); --g_buffers; return hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) {
  *e = reinterpret_cast<hipEvent_t>(new Event{g_device});
  ++g_events;
  return hipSuccess;
}
hipError_t hipEventDestroy(hipEvent_t e) { delete reinterpret_cast<Event *>(e); --g_events; return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t e, hipStream_t s) {
  return reinterpret_cast<Event *>(e)->device == device_of(s) ? hipSuccess : hipErrorInvalidHandle;
}
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipGetLastError() { return hipSuccess; }
hipError_t hipPointerGetAttributes(hipPointerAttribute_t *a, const void *p) {
  if (p == g_pinned) {
    a->type = hipMemoryTypeHost;
    return hipSuccess;
  }
  a->type = hipMemoryTypeUnregistered;
  return g_refuse_unknown ? hipErrorInvalidValue : hipSuccess;
}
hipError_t hipMemcpyAsync(void *dst, const void *src, size_t n, hipMemcpyKind, hipStream_t) {
  if (--g_fail_after < 0) return hipErrorUnknown;
  if (dst == g_pinned) ++g_direct;
  std::memcpy(dst, src, n);
  return hipSuccess;
}
}

static int check(bool ok, const char *what) {
  if (!ok) std::printf("FAILED: %s\n", what);
  return ok ? 0 : 1;
}

// a download of n bytes in two parts, as outputs are
static bool round_trip(fmmh::HostStageUser &user, int device, size_t n) {
  std::vector<char> a(n / 4), b(n - n / 4), x(a.size()), y(b.size());
  for (size_t i = 0; i < a.size(); ++i) a[i] = char(i * 7 + n);
  for (size_t i = 0; i < b.size(); ++i) b[i] = char(i * 11 + n);
  user.download(device, stream_of(device), {{x.data(), a.data(), a.size()}, {y.data(), b.data(), b.size()}});
  return a == x && b == y;
}
"""

DEVICES = r"""
int main() {
  int bad = 0;
  {
    fmmh::HostStageUser first, second;
    // operators of two devices in turn, from a thread whose device is the last one built
    hipSetDevice(1);
    for (size_t n : {1000u, 70000u, 300001u, 9000000u, 20000001u})
      for (int device : {0, 1, 0}) {
        bad += check(round_trip(device ? second : first, device, n), "round trip");
        bad += check(g_device == 1, "the caller's device is kept");
      }
    // a copy that fails: reported, the device kept, the next download as before
    hipSetDevice(1);
    g_fail_after = 2;
    bool thrown = false;
    try {
      round_trip(first, 0, 20000001);
    } catch (const std::runtime_error &) {
      thrown = true;
    }
    g_fail_after = 1 << 30;
    bad += check(thrown && g_device == 1, "a failed copy");
    bad += check(round_trip(first, 0, 20000001), "after a failed copy");
    // many threads: every buffer past the kept ones goes back at once
    std::vector<std::thread> work;
    std::atomic<int> wrong{0};
    for (int k = 0; k < 24; ++k)
      work.emplace_back([&, k] {
        for (int r = 0; r < 4; ++r) wrong += !round_trip(first, k & 1, 3000000 + k);
      });
    for (auto &t : work) t.join();
    bad += check(wrong == 0, "many threads");
    bad += check(g_buffers <= 8, "buffers kept");
  }
  bad += check(g_buffers == 0 && g_events == 0, "given back with the last user");
  return bad;
}
"""

PINNED = r"""
int main() {
  int bad = 0;
  fmmh::HostStageUser user;
  std::vector<char> a(3000000, 5), x(a.size());
  g_pinned = x.data();
  user.download(0, stream_of(0), {{x.data(), a.data(), a.size()}});
  bad += check(a == x && g_direct == 1 && g_buffers == 0, "memory the runtime knows takes one copy");
  g_pinned = nullptr;
  for (bool refuse : {false, true}) {
    g_refuse_unknown = refuse;
    bad += check(round_trip(user, 0, 3000000) && g_buffers == 1, "other memory is staged");
  }
  return bad;
}
"""

THREADS = r"""
#include <chrono>
#include <condition_variable>
#include <dirent.h>
#include <mutex>
static int threads() {
  int n = 0;
  DIR *d = opendir("/proc/self/task");
  while (dirent *e = readdir(d)) n += e->d_name[0] != '.';
  closedir(d);
  return n;
}
int main() {
  int bad = 0;
  const int before = threads();
  {
    fmmh::HostStageUser user;
    // callers that have downloaded and live on: at most four have kept threads of their own
    std::mutex mu;
    std::condition_variable cv;
    bool stop = false;
    int ready = 0;
    std::atomic<int> wrong{0};
    std::vector<std::thread> work;
    for (int k = 0; k < 20; ++k)
      work.emplace_back([&, k] {
        for (size_t n : {3000000u, 100000u, 9000001u}) wrong += !round_trip(user, k & 1, n + k);
        std::unique_lock<std::mutex> lock(mu);
        ++ready;
        cv.notify_all();
        cv.wait(lock, [&] { return stop; });
      });
    {
      std::unique_lock<std::mutex> lock(mu);
      cv.wait(lock, [&] { return ready == 20; });
      bad += check(threads() <= before + 20 + 4 * 7, "threads that stay");
      stop = true;
    }
    cv.notify_all();
    for (auto &t : work) t.join();
    bad += check(wrong == 0, "many threads");
  }
  for (int k = 0; k < 200 && threads() > before; ++k) std::this_thread::sleep_for(std::chrono::milliseconds(10));
  bad += check(threads() == before, "threads given back with the callers'");
  // and others may have them now
  fmmh::HostStageUser user;
  bad += check(round_trip(user, 0, 9000001), "another user");
  return bad;
}
"""


def _build(tmp_path, main):
    if shutil.which("g++") is None:
        pytest.skip("no g++")
    csrc = os.path.join(ROOT, "fmm_amd", "csrc")
    src = tmp_path / "t.cpp"
    src.write_text(RUNTIME + main)
    exe = tmp_path / "t"
    subprocess.run(["g++", "-std=c++17", "-O1", "-fopenmp", "-pthread", "-D__HIP_PLATFORM_AMD__", "-I" + csrc,
                    "-isystem/opt/rocm/include", str(src), os.path.join(csrc, "hoststage.cpp"), "-o", str(exe)],
                   check=True)
    return exe


def _run(exe, **env):
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=120, env={**os.environ, **env})
    assert r.returncode == 0, r.stdout + r.stderr


def test_downloads_of_several_devices(tmp_path):
    _run(_build(tmp_path, DEVICES))


def test_downloads_into_pinned_memory(tmp_path):
    _run(_build(tmp_path, PINNED))


def test_copying_threads_are_bounded(tmp_path):
    exe = _build(tmp_path, THREADS)
    _run(exe, OMP_NUM_THREADS="8")
    _run(exe, OMP_NUM_THREADS="1")
