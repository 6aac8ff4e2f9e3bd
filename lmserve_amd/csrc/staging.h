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
// handed out again once all have. Bounded: kStageSlots buffers of the largest size
// asked for (rounded up to a power of two). A thread that ends leaves its ring to
// the next one that needs a ring; kvc_thread_release frees the caller's and those.
constexpr int kStageSlots = 4;
constexpr int kStageMaxWgs = 64;
constexpr int64_t kStageHead = kStageMaxWgs * (int64_t)sizeof(uint32_t);

struct StageRing {
  char* base = nullptr;
  int64_t slot_bytes = 0;  // head included
  int next = 0;
  uint32_t seq = 0;
  uint32_t used_seq[kStageSlots] = {};
  int used_wgs[kStageSlots] = {};     // workgroups of the last kernel that read the slot, 0 = none
  int used_device[kStageSlots] = {};  // the device it runs on
  int64_t acquired = -1;              // bytes of the slot that is being filled, -1 = none
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

// Wait until the last reader of slot i is through. It normally has been for several
// calls; one that is still queued behind long work is waited for by looking at its
// words now and then, which holds up no other stream, thread or recording. Words that
// stay unset for a minute belong to a device that is in trouble, or to work that is
// very long indeed: the wait is then handed to that device, which says which.
int stage_wait(StageRing& r, int i) {
  if (!r.used_wgs[i]) return KVC_OK;
  const uint32_t* flags = reinterpret_cast<const uint32_t*>(r.base + i * r.slot_bytes);
  const auto read = [&] {
    for (int w = 0; w < r.used_wgs[i]; ++w)
      if (__atomic_load_n(flags + w, __ATOMIC_ACQUIRE) != r.used_seq[i]) return false;
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
    KVC_HIP(hipSetDevice(r.used_device[i]));
    const hipError_t e = hipDeviceSynchronize();
    KVC_HIP(hipSetDevice(dev));
    KVC_HIP(e);
  }
  r.used_wgs[i] = 0;
  return KVC_OK;
}

// the buffers of one ring, once nothing reads them
int stage_free(StageRing& r) {
  if (!r.base) return KVC_OK;
  for (int i = 0; i < kStageSlots; ++i) {
    const int rc = stage_wait(r, i);
    if (rc != KVC_OK) return rc;
  }
  char* base = r.base;
  r.base = nullptr;
  r.slot_bytes = 0;
  r.next = 0;
  r.acquired = -1;
  KVC_HIP(hipHostFree(base));
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
    const int rc_one = stage_free(*r);
    if (rc_one != KVC_OK) rc = rc_one;
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
      return fail(KVC_ERR_HIP, "kvc_staging_acquire: out of host memory");
    }
  }
  StageRing& r = *g_stage.ring;
  r.acquired = -1;
  if (kStageHead + bytes > r.slot_bytes) {
    int64_t slot = 64 << 10;
    while (slot < kStageHead + bytes) slot *= 2;
    const int rc = stage_free(r);
    if (rc != KVC_OK) return rc;
    void* base = nullptr;  // coherent: the words are polled while kernels run
    KVC_HIP(hipHostMalloc(&base, kStageSlots * slot, hipHostMallocPortable | hipHostMallocMapped | hipHostMallocCoherent));
    r.base = (char*)base;
    r.slot_bytes = slot;
    for (int i = 0; i < kStageSlots; ++i) std::memset(r.base + i * slot, 0, kStageHead);
  }
  const int rc = stage_wait(r, r.next);
  if (rc != KVC_OK) return rc;
  r.acquired = bytes;
  *out = r.base + r.next * r.slot_bytes + kStageHead;
  return KVC_OK;
}

// The acquired slot's flags and value for a kernel of `wgs` workgroups that reads it; the slot counts as in use
// from here on.
int stage_hand_over(const char* fn, int64_t bytes, int wgs, void* stream, uint32_t** flags, uint32_t* value) {
  StageRing* ring = g_stage.ring;
  if (!ring || ring->acquired < bytes)
    return fail(KVC_ERR_STAGING, "%s: %lld bytes wanted of a staging buffer of %lld (kvc_staging_acquire comes first)",
                fn, (long long)bytes, ring ? (long long)ring->acquired : -1ll);
  StageRing& r = *ring;
  hipStreamCaptureStatus capturing = hipStreamCaptureStatusNone;
  KVC_HIP(hipStreamIsCapturing((hipStream_t)stream, &capturing));
  if (capturing != hipStreamCaptureStatusNone)
    return fail(KVC_ERR_UNSUPPORTED, "%s: the staging buffer of a recorded launch would be overwritten before a replay", fn);
  const int i = r.next;
  KVC_HIP(hipGetDevice(&r.used_device[i]));
  if (++r.seq == 0) r.seq = 1;
  r.used_seq[i] = *value = r.seq;
  r.used_wgs[i] = wgs;
  *flags = reinterpret_cast<uint32_t*>(r.base + i * r.slot_bytes);
  r.next = (i + 1) % kStageSlots;
  r.acquired = -1;
  return KVC_OK;
}

// What the launch after a hand-over came to: a kernel that never started sets no words.
int stage_launched() {
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) {
    StageRing& r = *g_stage.ring;
    r.used_wgs[(r.next + kStageSlots - 1) % kStageSlots] = 0;
  }
  KVC_HIP(e);
  return KVC_OK;
}

}  // namespace
}  // namespace kvc

#endif  // KVC_STAGING_H_
