// rapt_copy.hip -- device to host copies of large results.
//
// The runtime copies to pageable memory through a pinned buffer with one host
// thread, which for a result array that is touched for the first time is bound
// by that thread's page faults (86 MB of trajectories: 9 ms, 9.5 GB/s).  Here the
// same staging has several threads behind it: the copy engine fills CHUNK-sized
// slots of a pinned ring in order, and each thread takes the next filled slot to
// its place in the result (2.5 ms, 34 GB/s; the link alone 57).
#include <hip/hip_runtime.h>
#include <stdint.h>
#include <string.h>

#include <atomic>
#include <thread>

#include "rapt_internal.hpp"

static constexpr size_t CHUNK = (size_t)1 << 20;
static constexpr int THREADS = 4;
// Below this the threads' start (about 20 us each) is not made up for.
static constexpr size_t COPY_MIN = (size_t)4 << 20;

static bool ring_make(rapt_ctx* c) {
  if (c->ring) return true;
  for (int i = 0; i < RAPT_RING_SLOTS; ++i)
    if (!c->ring_ev[i] &&
        hipEventCreateWithFlags(&c->ring_ev[i], hipEventDisableTiming) != hipSuccess)
      return false;
  void* p = nullptr;
  if (hipHostMalloc(&p, CHUNK * RAPT_RING_SLOTS, hipHostMallocDefault) != hipSuccess)
    return false;
  c->ring = static_cast<char*>(p);
  return true;
}

void rapt_ring_free(rapt_ctx* c) {
  if (c->ring) (void)hipHostFree(c->ring);
  c->ring = nullptr;
  for (hipEvent_t& e : c->ring_ev) {
    if (e) (void)hipEventDestroy(e);
    e = nullptr;
  }
}

// Memory that the runtime knows (pinned, managed or a device's) takes the copy
// as it is: PINNED.
static bool known_to_runtime(const void* p) {
  hipPointerAttribute_t a;
  if (hipPointerGetAttributes(&a, p) != hipSuccess) {
    (void)hipGetLastError();
    return false;
  }
  return a.type != hipMemoryTypeUnregistered;
}

hipError_t rapt_copy_out(rapt_ctx* c, void* dst, const void* src, size_t bytes) {
  if (bytes < COPY_MIN || known_to_runtime(dst))
    return hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToHost, c->stream);
  std::lock_guard<std::mutex> lock(c->ring_mu);  // one copy at a time has the ring
  if (!ring_make(c)) {
    (void)hipGetLastError();
    return hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToHost, c->stream);
  }
  constexpr size_t S = RAPT_RING_SLOTS;
  const size_t n = (bytes + CHUNK - 1) / CHUNK;
  std::atomic<size_t> filled{0}, next{0}, freed[S];  // freed: times a slot was emptied
  std::atomic<bool> stop{false};
  for (auto& f : freed) f.store(0, std::memory_order_relaxed);
  auto length = [&](size_t k) { return k + 1 < n ? CHUNK : bytes - k * CHUNK; };
  auto take = [&](size_t k) {
    memcpy(static_cast<char*>(dst) + k * CHUNK, c->ring + k % S * CHUNK, length(k));
    freed[k % S].store(k / S + 1, std::memory_order_release);
  };
  auto work = [&]() {
    for (size_t k; (k = next.fetch_add(1)) < n; take(k))
      while (filled.load(std::memory_order_acquire) <= k) {
        if (stop.load(std::memory_order_acquire)) return;
        std::this_thread::yield();
      }
  };
  std::thread th[THREADS];
  int started = 0;
  try {
    for (; started < THREADS; ++started) th[started] = std::thread(work);
  } catch (...) {  // no more threads: the ones there are, or this one, copy
  }
  hipError_t e = hipSuccess;
  size_t issued = 0;
  for (size_t k = 0; k < n && e == hipSuccess; ++k) {
    // every slot that is free, and chunk k's at least
    while (issued < n && e == hipSuccess) {
      if (freed[issued % S].load(std::memory_order_acquire) < issued / S) {
        if (issued > k) break;
        std::this_thread::yield();
        continue;
      }
      e = hipMemcpyAsync(c->ring + issued % S * CHUNK,
                         static_cast<const char*>(src) + issued * CHUNK, length(issued),
                         hipMemcpyDeviceToHost, c->stream);
      if (e == hipSuccess) e = hipEventRecord(c->ring_ev[issued % S], c->stream);
      ++issued;
    }
    if (e == hipSuccess) e = hipEventSynchronize(c->ring_ev[k % S]);
    if (e == hipSuccess) {
      filled.store(k + 1, std::memory_order_release);
      if (started == 0) take(k);
    }
  }
  if (e != hipSuccess) {
    stop.store(true, std::memory_order_release);
    (void)hipStreamSynchronize(c->stream);  // (nothing copies into the ring any more)
  }
  for (int i = 0; i < started; ++i) th[i].join();
  return e;
}
