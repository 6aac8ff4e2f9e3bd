// Staging of a step's inputs in pinned host memory (part of kvcache.hip; host code only).
#ifndef KVC_STAGING_H_
#define KVC_STAGING_H_

#include <hip/hip_runtime_api.h>

#include <chrono>
#include <cstdint>
#include <cstring>
#include <mutex>
#include <new>
#include <thread>

#include "common.h"

namespace kvc {
namespace {

// A ring of pinned buffers per thread in which a binding assembles what a small
// kernel then reads over the link itself: no copy command, no event (a recorded
// event costs 3 us of host time here, a launch 3). Each workgroup of the reading
// kernel sets a word in the buffer's head when it has read its share; a buffer is
// handed out again once all have. A buffer that is too small is replaced, its
// reader queued or not, by one of the next power of two; the outgrown one is kept
// until kvc_thread_release, because freeing pinned memory synchronises the device.
// So a thread holds kStageSlots times twice the largest size it asked for at most.
// A thread that ends leaves its ring to the next one that needs a ring;
// kvc_thread_release frees the caller's and those.
constexpr int kStageSlots = 4;
constexpr int kStageMaxWgs = 64;
constexpr int64_t kStageHead = kStageMaxWgs * (int64_t)sizeof(uint32_t);

struct StageBuffer {
  char* base = nullptr;
  int64_t bytes = 0;  // head included
  uint32_t used_seq = 0;
  int used_wgs = 0;     // workgroups of the last kernel that read it, 0 = none
  int used_device = 0;  // the device it runs on
  StageBuffer* next = nullptr;  // of the outgrown ones
};

struct StageRing {
  StageBuffer slot[kStageSlots];
  StageBuffer* outgrown = nullptr;
  int next = 0;
  uint32_t seq = 0;
  int64_t acquired = -1;  // bytes of the slot that is being filled, -1 = none
  StageRing* idle_next = nullptr;
};

std::mutex g_stage_mutex;
StageRing* g_stage_idle = nullptr;  // rings of threads that have ended, readers possibly still queued

struct StageHolder {
  StageRing* ring = nullptr;
  ~StageHolder() {  // no HIP call here: the process may be ending
    if (!ring) return;
    std::lock_guard<std::mutex> hold(g_stage_mutex);
    ring->acquired = -1;
    ring->idle_next = g_stage_idle;
    g_stage_idle = ring;
  }
};
thread_local StageHolder g_stage;

// Wait until the last reader of a buffer is through. It normally has been for several
// calls; one that is still queued behind long work is waited for by looking at its
// words now and then, which holds up no other stream, thread or recording. Words that
// stay unset for a minute belong to a device that is in trouble, or to work that is
// very long indeed: the wait is then handed to that device, which says which.
int stage_wait(StageBuffer& b) {
  if (!b.used_wgs) return KVC_OK;
  const uint32_t* flags = reinterpret_cast<const uint32_t*>(b.base);
  const auto read = [&] {
    for (int w = 0; w < b.used_wgs; ++w)
      if (__atomic_load_n(flags + w, __ATOMIC_ACQUIRE) != b.used_seq) return false;
    return true;
  };
  bool done = false;
  for (int spin = 0; spin < 2000 && !done; ++spin) done = read();
  for (int nap = 0; nap < 1000000 && !done; ++nap) {
    std::this_thread::sleep_for(std::chrono::microseconds(20));
    done = read();
  }
  if (!done) {
    int dev = 0;
    KVC_HIP(hipGetDevice(&dev));
    KVC_HIP(hipSetDevice(b.used_device));
    const hipError_t e = hipDeviceSynchronize();
    KVC_HIP(hipSetDevice(dev));
    KVC_HIP(e);
  }
  b.used_wgs = 0;
  return KVC_OK;
}

// a buffer, once nothing reads it
int stage_free(StageBuffer& b) {
  if (!b.base) return KVC_OK;
  const int rc = stage_wait(b);
  if (rc != KVC_OK) return rc;
  char* base = b.base;
  b.base = nullptr;
  b.bytes = 0;
  KVC_HIP(hipHostFree(base));
  return KVC_OK;
}

// A larger buffer in the place of one that its last reader may still be reading
int stage_grow(StageRing& r, StageBuffer& b, int64_t need) {
  int64_t bytes = 64 << 10;
  while (bytes < need) bytes *= 2;
  StageBuffer* old = nullptr;
  if (b.base && !(old = new (std::nothrow) StageBuffer))
    return fail(KVC_ERR_STAGING, "kvc_staging_acquire: out of host memory");
  void* base = nullptr;  // coherent: the words are polled while kernels run
  const hipError_t e = hipHostMalloc(&base, bytes, hipHostMallocPortable | hipHostMallocMapped | hipHostMallocCoherent);
  if (e != hipSuccess) {  // the caller has a path without staging: no error may stay behind for its next call
    delete old;
    (void)hipGetLastError();
    return fail(KVC_ERR_STAGING, "kvc_staging_acquire: no %lld bytes of pinned memory (%s)", (long long)bytes,
                hipGetErrorString(e));
  }
  std::memset(base, 0, kStageHead);
  if (old) {
    *old = b;
    old->next = r.outgrown;
    r.outgrown = old;
  }
  b = StageBuffer{};
  b.base = (char*)base;
  b.bytes = bytes;
  return KVC_OK;
}

int stage_release() {
  StageRing* mine = g_stage.ring;
  g_stage.ring = nullptr;
  StageRing* all;
  {
    std::lock_guard<std::mutex> hold(g_stage_mutex);
    all = g_stage_idle;
    g_stage_idle = nullptr;
  }
  if (mine) {
    mine->idle_next = all;
    all = mine;
  }
  int rc = KVC_OK;
  while (all) {
    StageRing* r = all;
    all = r->idle_next;
    const auto release = [&](StageBuffer& b) {
      const int rc_one = stage_free(b);
      if (rc_one != KVC_OK) rc = rc_one;
    };
    for (StageBuffer& b : r->slot) release(b);
    while (StageBuffer* b = r->outgrown) {
      r->outgrown = b->next;
      release(*b);
      delete b;
    }
    delete r;
  }
  return rc;
}

int stage_acquire(int64_t bytes, void** out) {
  *out = nullptr;
  if (!g_stage.ring) {
    std::lock_guard<std::mutex> hold(g_stage_mutex);
    if (g_stage_idle) {
      g_stage.ring = g_stage_idle;
      g_stage_idle = g_stage_idle->idle_next;
    } else if (!(g_stage.ring = new (std::nothrow) StageRing)) {
      return fail(KVC_ERR_STAGING, "kvc_staging_acquire: out of host memory");
    }
  }
  StageRing& r = *g_stage.ring;
  r.acquired = -1;
  StageBuffer& b = r.slot[r.next];
  const int rc = kStageHead + bytes > b.bytes ? stage_grow(r, b, kStageHead + bytes) : stage_wait(b);
  if (rc != KVC_OK) return rc;
  r.acquired = bytes;
  *out = b.base + kStageHead;
  return KVC_OK;
}

// The acquired slot's flags and value for a kernel of `wgs` workgroups that reads it; the slot counts as in use
// from here on.
int stage_hand_over(const char* fn, int64_t bytes, int wgs, void* stream, uint32_t** flags, uint32_t* value) {
  StageRing* ring = g_stage.ring;
  if (!ring || ring->acquired < bytes)
    return fail(KVC_ERR_STAGING, "%s: %lld bytes wanted of a staging buffer of %lld (kvc_staging_acquire comes first)",
                fn, (long long)bytes, ring ? (long long)ring->acquired : -1ll);
  // an error that an earlier call of the application left: stage_launched would take it for the launch's own, and
  // the buffer for free while the kernel reads it
  KVC_HIP(hipGetLastError());
  StageRing& r = *ring;
  hipStreamCaptureStatus capturing = hipStreamCaptureStatusNone;
  KVC_HIP(hipStreamIsCapturing((hipStream_t)stream, &capturing));
  if (capturing != hipStreamCaptureStatusNone)
    return fail(KVC_ERR_UNSUPPORTED, "%s: the staging buffer of a recorded launch would be overwritten before a replay", fn);
  StageBuffer& b = r.slot[r.next];
  KVC_HIP(hipGetDevice(&b.used_device));
  if (++r.seq == 0) r.seq = 1;
  b.used_seq = *value = r.seq;
  b.used_wgs = wgs;
  *flags = reinterpret_cast<uint32_t*>(b.base);
  r.next = (r.next + 1) % kStageSlots;
  r.acquired = -1;
  return KVC_OK;
}

// What the launch after a hand-over came to: a kernel that never started sets no words.
int stage_launched() {
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) {
    StageRing& r = *g_stage.ring;
    r.slot[(r.next + kStageSlots - 1) % kStageSlots].used_wgs = 0;
  }
  KVC_HIP(e);
  return KVC_OK;
}

}  // namespace
}  // namespace kvc

#endif  // KVC_STAGING_H_
