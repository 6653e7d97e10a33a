// host_copy.hpp -- large copies between device memory and ordinary (pageable)
// host arrays.
//
// hipMemcpy stages such a copy through one CPU thread: on an MI355X host it
// reached 10 GB/s into a freshly allocated array (its pages are touched for the
// first time by that thread), 16 GB/s into a used one and 27 GB/s to the
// device, against 57 GB/s of the link from pinned memory.  Here the link moves
// chunks between the device and a ring of pinned buffers while up to 8 threads
// move them between the ring and the caller's array.  Measured, 1.02 GB: 98 ->
// 24 ms into a fresh array (43 GB/s), 58 -> 20 ms into a used one, 34 -> 22 ms to
// the device (45 GB/s).
#pragma once
#include <hip/hip_runtime.h>
#include <sched.h>

#include <algorithm>
#include <atomic>
#include <cstring>
#include <memory>
#include <mutex>
#include <new>
#include <thread>
#include <vector>

namespace hostcopy {

constexpr size_t CHUNK = (size_t)4 << 20;  // the largest chunk, one buffer of the ring
constexpr int NBUF = 8;                    // 32 MiB of pinned memory in all
constexpr int LAG = 4;                     // chunks on the link before the oldest is waited for
constexpr int WORKERS = 8;                 // at most: see workers()
// Smaller copies are left to hipMemcpy: starting the threads costs about 0.1 ms
// (to the host 4.7 MB 0.28 / 0.28 ms, 9.4 MB 0.57 -> 0.37; to the device 9.4 MB
// 0.29 -> 0.42, where hipMemcpy itself reaches 29-32 GB/s, 201 MB 7.0 -> 4.7).
constexpr size_t MIN_TO_HOST = (size_t)4 << 20, MIN_TO_DEVICE = (size_t)64 << 20;
// An eighth of a small copy a chunk, so that the threads start early; 4 MiB of
// a large one, because each chunk costs the link about 15 us beside its bytes
// (1 GiB to a fresh array, moved by hipMemcpyAsync: 30, 38 and 43 GB/s with chunks
// of 1, 2 and 4 MiB).
constexpr size_t MIN_CHUNK = (size_t)512 << 10;

// The pinned ring: one for the process, kept while any handle is alive.  A
// second thread that wants it meanwhile copies without it.
struct Ring {
  std::mutex mu;
  int users = 0;
  char* pin = nullptr;
};
inline Ring& ring() {
  static Ring r;
  return r;
}
inline void retain() {
  std::lock_guard<std::mutex> l(ring().mu);
  ++ring().users;
}
inline void release() {
  Ring& r = ring();
  std::lock_guard<std::mutex> l(r.mu);
  if (--r.users == 0 && r.pin) {
    (void)hipHostFree(r.pin);
    r.pin = nullptr;
  }
}

// Threads of a copy: one for each core that the caller may run on beside its own,
// since threads that wait do so on the core (a waiting thread that sleeps would
// be woken for every chunk of 0.1 ms).  0, a single core: hipMemcpy's one thread.
inline int workers() {
  cpu_set_t set;
  const int n = sched_getaffinity(0, sizeof set, &set) == 0
                    ? CPU_COUNT(&set)
                    : (int)std::thread::hardware_concurrency();
  return std::max(0, std::min(WORKERS, n - 1));
}

// (to the device: in order on st, whose work the callers wait for before they
// return to their own)
inline hipError_t direct(void* dev, void* host, size_t bytes, bool to_host, hipStream_t st) {
  if (!to_host) return hipMemcpyAsync(dev, host, bytes, hipMemcpyHostToDevice, st);
  const hipError_t e = hipMemcpyAsync(host, dev, bytes, hipMemcpyDeviceToHost, st);
  return e != hipSuccess ? e : hipStreamSynchronize(st);
}

// whether the runtime knows the host array (pinned: hipMemcpy is at the link's
// rate by itself)
inline bool pinned(const void* host) {
  hipPointerAttribute_t a;
  if (hipPointerGetAttributes(&a, host) == hipSuccess) return a.type != hipMemoryTypeUnregistered;
  (void)hipGetLastError();  // an unknown address is not an error here
  return false;
}

// bytes of device memory into a pinned buffer, by a kernel (dwf_gpu.hip).  Not
// hipMemcpyAsync: that is the DMA engine's, and with an event behind each copy
// the engine and the stream's queue wait for each other, 25 us a chunk and, in
// phases such as the 30 ms after a batched operator call, 130 us (copy trace; the
// copy of 0.7 MB itself takes 17).  5.8 MB to the host 0.36 and, in such a phase,
// 1.26 ms, where one hipMemcpy took 0.35; 151 MB 8.0 ms.  By kernel 0.29 and 3.2
// ms, in either state.
__attribute__((visibility("hidden"))) hipError_t to_pinned(void* pin, const void* dev,
                                                          size_t bytes, hipStream_t st);

// dev <-> host, after the work queued on st; to the host complete on return
inline hipError_t copy(void* dev, void* host, size_t bytes, bool to_host, hipStream_t st) {
  if (bytes < (to_host ? MIN_TO_HOST : MIN_TO_DEVICE) || pinned(host))
    return direct(dev, host, bytes, to_host, st);
  const int nworker = workers();
  Ring& r = ring();
  std::unique_lock<std::mutex> own(r.mu, std::try_to_lock);
  if (nworker == 0 || !own.owns_lock()) return direct(dev, host, bytes, to_host, st);
  if (!r.pin && hipHostMalloc((void**)&r.pin, NBUF * CHUNK, hipHostMallocPortable) != hipSuccess) {
    (void)hipGetLastError();
    r.pin = nullptr;
    return direct(dev, host, bytes, to_host, st);
  }
  const size_t chunk = std::min(CHUNK, std::max(MIN_CHUNK, (bytes / 8 + 4095) / 4096 * 4096));
  const size_t n = (bytes + chunk - 1) / chunk;
  std::unique_ptr<std::atomic<bool>[]> moved(new (std::nothrow) std::atomic<bool>[n]);
  if (!moved) return direct(dev, host, bytes, to_host, st);
  for (size_t t = 0; t < n; ++t) moved[t].store(false, std::memory_order_relaxed);
  struct Events {  // of the stream's device, so made per copy
    hipEvent_t e[NBUF] = {};
    ~Events() {
      for (auto x : e)
        if (x) (void)hipEventDestroy(x);
    }
  } ev;
  for (auto& x : ev.e) {
    const hipError_t e = hipEventCreateWithFlags(&x, hipEventDisableTiming);
    if (e != hipSuccess) return e;
  }
  // `gate`: chunks a worker may move: those the link has delivered (to host),
  // or those whose buffer the link has emptied (to device)
  std::atomic<size_t> next{0}, gate{to_host ? 0 : (size_t)NBUF};
  std::atomic<bool> stop{false};
  char* const pin = r.pin;
  auto len = [&](size_t t) { return t + 1 < n ? chunk : bytes - t * chunk; };
  auto worker = [&]() {
    for (size_t t; (t = next.fetch_add(1)) < n;) {
      while (gate.load(std::memory_order_acquire) <= t) {
        if (stop.load(std::memory_order_relaxed)) return;
        std::this_thread::yield();
      }
      char *p = pin + (t % NBUF) * CHUNK, *q = (char*)host + t * chunk;
      if (to_host)
        std::memcpy(q, p, len(t));
      else
        std::memcpy(p, q, len(t));
      moved[t].store(true, std::memory_order_release);
    }
  };
  std::thread pool[WORKERS];
  int started = 0;
  try {
    for (; started < nworker; ++started) pool[started] = std::thread(worker);
  } catch (...) {  // fewer threads than asked for
  }
  hipError_t err = hipSuccess;
  if (started == 0) {
    err = direct(dev, host, bytes, to_host, st);
  } else {
    auto wait = [&](size_t t) {
      while (!moved[t].load(std::memory_order_acquire)) std::this_thread::yield();
    };
    for (size_t t = 0; t < n + LAG && err == hipSuccess; ++t) {
      if (t < n) {
        if (to_host ? t >= NBUF : true) wait(to_host ? t - NBUF : t);
        char *p = pin + (t % NBUF) * CHUNK, *d = (char*)dev + t * chunk;
        err = to_host ? to_pinned(p, d, len(t), st)
                      : hipMemcpyAsync(d, p, len(t), hipMemcpyHostToDevice, st);
        if (err == hipSuccess) err = hipEventRecord(ev.e[t % NBUF], st);
      }
      if (t >= LAG && err == hipSuccess) {
        err = hipEventSynchronize(ev.e[(t - LAG) % NBUF]);
        gate.store(t - LAG + 1 + (to_host ? 0 : NBUF), std::memory_order_release);
      }
    }
    if (err != hipSuccess) {
      stop.store(true);
      (void)hipStreamSynchronize(st);  // the link is done with the ring
    }
  }
  for (int k = 0; k < started; ++k) pool[k].join();
  return err;
}

}  // namespace hostcopy
