// Host transfers: large downloads into the caller's memory and the checks
// of uploaded positions.
#pragma once
#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <cmath>
#include <cstring>
#include <map>
#include <memory>
#include <mutex>
#include <system_error>
#include <thread>
#include <vector>

#include "mfe_internal.h"

namespace mfe {

// Download of results of some megabytes.  The caller's memory is pageable
// and, where it was just allocated, has no pages yet: the runtime's copy
// into it runs on one thread, page faults included.  Here the data go
// through a ring of pinned slots, and threads that live for the call copy
// each slot out.  Measured, runtime -> ring: positions, velocities and
// accelerations of a million particles into new arrays (72 MB) 5.4 -> 2.4 ms,
// of 200000 (14.4 MB) 1.07 -> 0.90 ms, into kept arrays 0.79 -> 0.53; forces
// of 100000 (2.4 MB) 0.171 -> 0.157 ms new, 0.149 -> 0.122 ms into kept
// arrays; below two slots nothing overlaps.
//
// The engines of a device share one ring, which the last of them frees.  The
// first touch of its pages costs the host 0.1 ms per MB with all threads
// (0.38 ms with one), so with a ring of its own every engine's first download
// had been slower than the runtime's wherever the caller's memory had pages:
// 3.6 MB 0.29 -> 1.0 ms, 14.4 MB 2.0 -> 2.6, now 0.24 and 0.95 from the second
// engine on.  (Leaving the first downloads to the runtime instead cost more
// where that memory had none: 14.4 MB 2.3 and 2.4 ms for the first two, 2.5
// and 0.9 through a new ring.)  A download that finds the ring in use by
// another engine's takes the runtime's copy.
struct DownloadRing {
  // half of a slot is used below kHalfBelow, where its copies are too few to
  // overlap (3.0 ms with half slots for the 72 MB)
  static constexpr size_t kSlot = 2 << 20, kHalfBelow = 16 << 20;
  static constexpr int kSlots = 16;
  // a slot is filled again this many chunks after its own, and may still be
  // being copied out until then; the rest of the ring is in flight
  static constexpr int kLag = 10;
  static constexpr int kThreads = 6;

  std::mutex mu;
  char *pin = nullptr;
  size_t bytes = 0;
  hipEvent_t ev[kSlots] = {};

  // the slot size of a download of `total` bytes, with the slots made
  size_t take(size_t total) {
    const size_t slot = total < kHalfBelow ? kSlot / 2 : kSlot;
    if (bytes >= kSlots * slot) return slot;
    for (hipEvent_t &x : ev)
      if (!x) MFE_HIP_TRY(hipEventCreateWithFlags(&x, hipEventDisableTiming));
    if (pin) MFE_HIP_TRY(hipHostFree(pin));
    pin = nullptr;
    bytes = 0;
    MFE_HIP_TRY(hipHostMalloc((void **)&pin, kSlots * slot));
    bytes = kSlots * slot;
    return slot;
  }
  ~DownloadRing() {
    if (pin) (void)hipHostFree(pin);
    for (hipEvent_t &x : ev)
      if (x) (void)hipEventDestroy(x);
  }
};

// the device's ring, shared by the engines that hold it
inline std::shared_ptr<DownloadRing> device_ring(int device) {
  static std::mutex mu;
  static std::map<int, std::weak_ptr<DownloadRing>> rings;
  std::lock_guard<std::mutex> turn(mu);
  std::shared_ptr<DownloadRing> r = rings[device].lock();
  if (!r) rings[device] = r = std::make_shared<DownloadRing>();
  return r;
}

constexpr size_t kDownloadRingMin = 2 << 20;

struct DownloadPart {
  void *dst;
  const void *src;  // device
  size_t bytes;
};

// the parts copied to the host; waits for the stream (wait false: the
// caller does, before it reads a small part)
inline void download(DownloadRing &ring, int device, const std::vector<DownloadPart> &parts,
                     hipStream_t s, bool wait = true) {
  size_t total = 0;
  for (const DownloadPart &p : parts) total += p.bytes;
  std::unique_lock<std::mutex> turn(ring.mu, std::defer_lock);
  size_t slot = 0;
  if (total >= kDownloadRingMin) {
    MFE_HIP_TRY(hipSetDevice(device));
    if (turn.try_lock()) slot = ring.take(total);
  }
  if (!slot) {
    for (const DownloadPart &p : parts)
      MFE_HIP_TRY(hipMemcpyAsync(p.dst, p.src, p.bytes, hipMemcpyDeviceToHost, s));
    if (wait) MFE_HIP_TRY(hipStreamSynchronize(s));
    return;
  }
  std::vector<DownloadPart> c;
  for (const DownloadPart &p : parts)
    for (size_t o = 0; o < p.bytes; o += slot)
      c.push_back({(char *)p.dst + o, (const char *)p.src + o, std::min(slot, p.bytes - o)});
  constexpr int K = DownloadRing::kSlots;
  const int n = (int)c.size();
  std::atomic<int> ready{0}, next{0}, stop{0};
  std::vector<std::atomic<int>> done(n);
  for (auto &d : done) d.store(0, std::memory_order_relaxed);
  auto copy_out = [&](int k) {
    std::memcpy(c[k].dst, ring.pin + (k % K) * slot, c[k].bytes);
    done[k].store(1, std::memory_order_release);
  };
  auto work = [&]() {
    for (;;) {
      const int k = next.fetch_add(1);
      if (k >= n) return;
      while (ready.load(std::memory_order_acquire) <= k) {
        if (stop.load(std::memory_order_relaxed)) return;
        std::this_thread::yield();
      }
      copy_out(k);
    }
  };
  // the threads end with the call and no copy into the slots outlives it,
  // also when one fails
  struct Ended {
    std::vector<std::thread> t;
    std::atomic<int> &stop;
    hipStream_t s;
    bool complete;
    ~Ended() {
      stop.store(1);
      for (std::thread &x : t) x.join();
      if (!complete) (void)hipStreamSynchronize(s);
    }
  } pool{{}, stop, s, false};
  pool.t.reserve(DownloadRing::kThreads);
  auto issue = [&](int k) {
    MFE_HIP_TRY(hipMemcpyAsync(ring.pin + (k % K) * slot, c[k].src, c[k].bytes,
                               hipMemcpyDeviceToHost, s));
    MFE_HIP_TRY(hipEventRecord(ring.ev[k % K], s));
  };
  for (int k = 0; k < std::min(n, K); ++k) issue(k);
  try {
    for (int k = 0; k < std::min(n / 2, DownloadRing::kThreads); ++k) pool.t.emplace_back(work);
  } catch (const std::system_error &) {
    // as many threads as the system gives
  }
  auto finished = [&](int k) {
    while (!done[k].load(std::memory_order_acquire)) std::this_thread::yield();
  };
  for (int k = 0; k < n; ++k) {
    MFE_HIP_TRY(hipEventSynchronize(ring.ev[k % K]));
    ready.store(k + 1, std::memory_order_release);
    if (pool.t.empty()) copy_out(k);
    const int old = k - DownloadRing::kLag;
    if (old >= 0 && old + K < n) {
      finished(old);
      issue(old + K);
    }
  }
  for (int k = 0; k < n; ++k) finished(k);
  pool.complete = true;
}

// whether every coordinate of n particles lies in the box [-L2, L2] (NaN
// does not), six coordinates at a time so that the compiler takes them in
// vectors: one by one, with the axis from the index modulo 3, took half of
// an upload of 100000 particles
inline bool in_box(const double *r, size_t n, const double L2[3]) {
  const double lim[6] = {L2[0], L2[1], L2[2], L2[0], L2[1], L2[2]};
  int ok[6] = {1, 1, 1, 1, 1, 1};
  size_t i = 0;
  for (; i + 2 <= n; i += 2)
    for (int m = 0; m < 6; ++m) ok[m] &= std::fabs(r[3 * i + m]) <= lim[m];
  if (i < n)
    for (int m = 0; m < 3; ++m) ok[m] &= std::fabs(r[3 * i + m]) <= lim[m];
  return ok[0] & ok[1] & ok[2] & ok[3] & ok[4] & ok[5];
}

}  // namespace mfe
