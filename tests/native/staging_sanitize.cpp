// The staging ring of a step's inputs against a runtime made of stubs: the driver plays the kernels that read the
// buffers by setting their words itself, now, later or never. Built with a sanitizer by tests/test_host_sanitizers.py.
#include <unistd.h>

#include <atomic>
#include <cstdarg>
#include <cstdio>
#include <cstdlib>
#include <map>
#include <mutex>
#include <thread>
#include <vector>

#include "staging.h"

namespace {
std::mutex g_mutex;
std::map<void*, size_t> g_pinned;  // live allocations
std::atomic<int> g_frees{0}, g_device_waits{0}, g_cleared{0};
std::atomic<bool> g_out_of_memory{false};
std::atomic<hipError_t> g_last_error{hipSuccess};

size_t pinned_bytes() {
  std::lock_guard<std::mutex> hold(g_mutex);
  size_t n = 0;
  for (const auto& a : g_pinned) n += a.second;
  return n;
}
}  // namespace

extern "C" {
hipError_t hipHostMalloc(void** p, size_t bytes, unsigned int) {
  if (g_out_of_memory) return hipErrorOutOfMemory;
  *p = calloc(1, bytes);
  std::lock_guard<std::mutex> hold(g_mutex);
  g_pinned[*p] = bytes;
  return hipSuccess;
}
hipError_t hipHostFree(void* p) {
  ++g_frees;
  std::lock_guard<std::mutex> hold(g_mutex);
  if (!g_pinned.erase(p)) return hipErrorInvalidValue;
  free(p);
  return hipSuccess;
}
hipError_t hipGetDevice(int* d) { return *d = 0, hipSuccess; }
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipDeviceSynchronize() { return ++g_device_waits, hipSuccess; }
hipError_t hipGetLastError() { return ++g_cleared, g_last_error.exchange(hipSuccess); }
hipError_t hipStreamIsCapturing(hipStream_t, hipStreamCaptureStatus* s) {
  return *s = hipStreamCaptureStatusNone, hipSuccess;
}
const char* hipGetErrorString(hipError_t) { return "stub"; }
}

namespace kvc {
int fail(int code, const char*, ...) { return code; }
}  // namespace kvc

namespace {
int bad = 0;
#define CHECK(x)                                              \
  do {                                                        \
    if (!(x)) {                                               \
      ++bad;                                                  \
      std::printf("line %d: %s\n", __LINE__, #x);             \
    }                                                         \
  } while (0)

struct Reader {  // a launch that reads a buffer with `wgs` workgroups
  uint32_t* flags = nullptr;
  uint32_t value = 0;
  int wgs = 0;
  char* data() const { return reinterpret_cast<char*>(flags) + kvc::kStageHead; }
  void done() const {
    for (int w = 0; w < wgs; ++w) __atomic_store_n(flags + w, value, __ATOMIC_RELEASE);
  }
};

Reader launch(int64_t bytes, int wgs, char mark) {
  Reader r;
  void* p = nullptr;
  CHECK(kvc::stage_acquire(bytes, &p) == KVC_OK);
  if (!p) exit(1);
  memset(p, mark, bytes);
  CHECK(kvc::stage_hand_over("driver", bytes, wgs, nullptr, &r.flags, &r.value) == KVC_OK);
  r.wgs = wgs;
  CHECK((char*)p == r.data());
  CHECK(kvc::stage_launched() == KVC_OK);
  return r;
}

bool holds(const Reader& r, int64_t bytes, char mark) {
  for (int64_t i = 0; i < bytes; ++i)
    if (r.data()[i] != mark) return false;
  return true;
}
}  // namespace

int main() {
  alarm(100);
  {  // larger steps while no reader of the smaller ones is through: nothing waits, nothing is freed, nothing is overwritten
    const auto t0 = std::chrono::steady_clock::now();
    std::vector<Reader> queued;
    std::vector<int64_t> sizes;
    for (int64_t bytes : {100, 200, 300, 400, 70000, 140000, 70000, 300000, 1 << 20}) {
      queued.push_back(launch(bytes, 1 + (int)queued.size(), (char)('a' + queued.size())));
      sizes.push_back(bytes);
    }
    CHECK(std::chrono::steady_clock::now() - t0 < std::chrono::seconds(10));
    CHECK(g_frees == 0 && g_device_waits == 0);
    for (size_t i = 0; i < queued.size(); ++i) CHECK(holds(queued[i], sizes[i], (char)('a' + i)));
    for (const Reader& r : queued) r.done();
    const size_t before = pinned_bytes();
    for (int k = 0; k < 40; ++k) launch(1 << 19, 3, 'z').done();  // grown slots are reused
    CHECK(pinned_bytes() <= before + 3 * (2 << 20));
    CHECK(kvc::stage_release() == KVC_OK);
    CHECK(pinned_bytes() == 0);
  }
  g_frees = 0;
  {  // what a thread ever holds is at most twice its largest buffers
    for (int64_t bytes = 1; bytes < (1 << 22); bytes *= 2)
      for (int k = 0; k < 4; ++k) launch(bytes, 64, 'b').done();
    CHECK(pinned_bytes() <= 4 * 2 * (size_t)(1 << 22));
    CHECK(g_frees == 0);
    CHECK(kvc::stage_release() == KVC_OK);
    CHECK(pinned_bytes() == 0);
  }
  {  // no pinned memory: said as such, no error left behind, and what the ring has stays in use
    Reader first = launch(100, 2, 'p');
    for (int k = 0; k < 3; ++k) launch(100, 1, 'q').done();
    void* p = nullptr;
    g_out_of_memory = true;
    g_cleared = 0;
    CHECK(kvc::stage_acquire(1 << 20, &p) == KVC_ERR_STAGING && p == nullptr && g_cleared == 1);
    CHECK(holds(first, 100, 'p'));
    first.done();
    CHECK(kvc::stage_acquire(200, &p) == KVC_OK && p == first.data());
    g_out_of_memory = false;
    launch(1 << 20, 1, 'r').done();
    CHECK(kvc::stage_release() == KVC_OK);
    CHECK(pinned_bytes() == 0);
    g_out_of_memory = true;
    CHECK(kvc::stage_acquire(100, &p) == KVC_ERR_STAGING);
    g_out_of_memory = false;
    launch(100, 1, 's').done();
    CHECK(kvc::stage_release() == KVC_OK);
  }
  {  // an error from before the launch is reported before it; one of the launch leaves the buffer free
    void* p = nullptr;
    uint32_t *flags = nullptr, value = 0;
    CHECK(kvc::stage_acquire(100, &p) == KVC_OK);
    g_last_error = hipErrorInvalidValue;
    CHECK(kvc::stage_hand_over("driver", 100, 1, nullptr, &flags, &value) == KVC_ERR_HIP);
    CHECK(kvc::stage_hand_over("driver", 100, 1, nullptr, &flags, &value) == KVC_OK);
    g_last_error = hipErrorInvalidConfiguration;
    CHECK(kvc::stage_launched() == KVC_ERR_HIP);
    for (int k = 0; k < 4; ++k) launch(100, 1, 't').done();
    CHECK(kvc::stage_release() == KVC_OK);
  }
  {  // threads that end: six of them come round to buffers that a reader of an ended thread still has
    std::vector<Reader> queued;
    std::vector<std::thread> devices;
    for (int k = 0; k < 6; ++k) {
      Reader r;
      double waited = 0;
      std::thread([&] {
        const auto t0 = std::chrono::steady_clock::now();
        r = launch(1000, 2, (char)('a' + k));
        waited = std::chrono::duration<double>(std::chrono::steady_clock::now() - t0).count();
      }).join();
      CHECK(k < 4 ? waited < 0.05 : waited > 0.02);
      if (k >= 3) {  // the oldest reader is through 60 ms from now
        const Reader oldest = queued[k - 3];
        const char mark = (char)('a' + k - 3);
        devices.emplace_back([oldest, mark] {
          std::this_thread::sleep_for(std::chrono::milliseconds(60));
          if (!holds(oldest, 1000, mark)) std::printf("overwritten\n"), exit(1);
          oldest.done();
        });
      }
      queued.push_back(r);
    }
    for (std::thread& d : devices) d.join();
    for (const Reader& r : queued) r.done();
    CHECK(kvc::stage_release() == KVC_OK);
    CHECK(pinned_bytes() == 0);
  }
  std::printf("bad=%d\n", bad);
  return bad != 0;
}
