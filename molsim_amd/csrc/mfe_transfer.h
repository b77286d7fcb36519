// Host transfers: large downloads into the caller's memory and the checks
// of uploaded positions.
#pragma once
#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <cmath>
#include <cstring>
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
// accelerations of a million particles into new arrays (72 MB) 6.7 -> 2.6 ms,
// of 200000 (14.4 MB) 0.99 -> 0.78 ms; forces of 100000 (2.4 MB) 0.171 ->
// 0.157 ms new, 0.149 -> 0.122 ms into kept arrays; below two slots nothing
// overlaps.
struct DownloadRing {
  // half of a slot is used below kHalfBelow, where its copies are too few to
  // overlap (3.0 ms with half slots for the 72 MB)
  static constexpr size_t kSlot = 2 << 20, kHalfBelow = 16 << 20;
  static constexpr int kSlots = 16;
  // a slot is filled again this many chunks after its own, and may still be
  // being copied out until then; the rest of the ring is in flight
  static constexpr int kLag = 10;
  static constexpr int kThreads = 6;

  std::mutex mu;  // downloads of one engine from several threads take turns
  char *pin = nullptr;
  size_t bytes = 0;
  hipEvent_t ev[kSlots] = {};

  // room for `need` bytes of slots (no more than a download has)
  void create(size_t need) {
    for (hipEvent_t &x : ev)
      if (!x) MFE_HIP_TRY(hipEventCreateWithFlags(&x, hipEventDisableTiming));
    if (bytes >= need) return;
    if (pin) MFE_HIP_TRY(hipHostFree(pin));
    pin = nullptr;
    bytes = 0;
    MFE_HIP_TRY(hipHostMalloc((void **)&pin, need));
    bytes = need;
  }
  void release() {
    if (pin) (void)hipHostFree(pin);
    pin = nullptr;
    bytes = 0;
    for (hipEvent_t &x : ev) {
      if (x) (void)hipEventDestroy(x);
      x = nullptr;
    }
  }
};

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
  if (total < kDownloadRingMin) {
    for (const DownloadPart &p : parts)
      MFE_HIP_TRY(hipMemcpyAsync(p.dst, p.src, p.bytes, hipMemcpyDeviceToHost, s));
    if (wait) MFE_HIP_TRY(hipStreamSynchronize(s));
    return;
  }
  MFE_HIP_TRY(hipSetDevice(device));
  std::lock_guard<std::mutex> turn(ring.mu);
  const size_t slot = total < DownloadRing::kHalfBelow ? DownloadRing::kSlot / 2
                                                       : DownloadRing::kSlot;
  std::vector<DownloadPart> c;
  for (const DownloadPart &p : parts)
    for (size_t o = 0; o < p.bytes; o += slot)
      c.push_back({(char *)p.dst + o, (const char *)p.src + o, std::min(slot, p.bytes - o)});
  constexpr int K = DownloadRing::kSlots;
  const int n = (int)c.size();
  ring.create(std::min(n, K) * slot);
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
  // the threads end with the call, also when a copy fails
  struct Joined {
    std::vector<std::thread> t;
    std::atomic<int> &stop;
    ~Joined() {
      stop.store(1);
      for (std::thread &x : t) x.join();
    }
  } pool{{}, stop};
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
