// smx_ring.h -- host transfers of whole fields (host code only).
//
// Through the runtime a 256^3 field (134 MB) takes 13.6 ms into a fresh array and 8 ms into a used one
// (one thread, which also takes the page faults) and 5.2 ms the other way.  Here a large field goes
// through a ring of pinned slots: each worker thread moves its own chunks between its two slots and the
// caller's array while the device copy of its other slot runs, 4.4, 3.6 and 4.0 ms.  Short of kRingToHost
// (96^3, 7 MB: 0.48 -> 0.38 ms; 64^3, 2 MB: 0.17 -> 0.22) and kRingToDevice bytes (25 MB: the same; 57 MB:
// 2.2 -> 1.8 ms) the runtime's copy is as fast.  One ring per process, used by one transfer at a time (another
// one, from another thread, takes the runtime's copy); allocated by the first large transfer (2 ms), freed
// with the last handle.
#pragma once
#include <hip/hip_runtime_api.h>

#include <algorithm>
#include <atomic>
#include <cstring>
#include <exception>
#include <mutex>
#include <thread>
#include <vector>

namespace smx {

constexpr size_t kRingSlot = 2u << 20;
constexpr size_t kRingToHost = 4u << 20, kRingToDevice = 32u << 20;
constexpr int kRingWorkers = 8, kRingSlots = 2 * kRingWorkers;
struct HostRing {
  std::mutex use;   // held by the transfer that uses buf
  std::mutex refs_mu;
  int refs = 0;
  char* buf = nullptr;
};
inline HostRing g_ring;
inline void ring_retain() {
  std::lock_guard<std::mutex> lk(g_ring.refs_mu);
  ++g_ring.refs;
}
inline void ring_release() {
  std::lock_guard<std::mutex> lk(g_ring.refs_mu);
  if (--g_ring.refs > 0) return;
  std::lock_guard<std::mutex> use(g_ring.use);
  if (g_ring.buf) (void)hipHostFree(g_ring.buf);
  g_ring.buf = nullptr;
}

// Chunks w, w + nw, ... of one transfer through two slots, on the handle's stream.
inline hipError_t ring_worker(int device, hipStream_t st, char* dev, char* host, size_t bytes, size_t chunk,
                              bool to_host, int w, int nw, char* slots) {
  hipError_t e = hipSetDevice(device);
  hipEvent_t ev[2] = {nullptr, nullptr};
  for (auto& x : ev)
    if (e == hipSuccess) e = hipEventCreateWithFlags(&x, hipEventDisableTiming);
  const size_t nchunks = (bytes + chunk - 1) / chunk;
  auto size = [&](size_t c) { return std::min(chunk, bytes - c * chunk); };
  auto issue = [&](size_t c, int s) {
    char* d = dev + c * chunk;
    char* b = slots + s * kRingSlot;
    e = to_host ? hipMemcpyAsync(b, d, size(c), hipMemcpyDeviceToHost, st)
                : hipMemcpyAsync(d, b, size(c), hipMemcpyHostToDevice, st);
    if (e == hipSuccess) e = hipEventRecord(ev[s], st);
  };
  int s = 0;
  if (to_host) {
    for (size_t c = w; c < nchunks && c < (size_t)w + 2 * nw && e == hipSuccess; c += nw, s ^= 1) issue(c, s);
    s = 0;
    for (size_t c = w; c < nchunks && e == hipSuccess; c += nw, s ^= 1) {
      e = hipEventSynchronize(ev[s]);
      if (e != hipSuccess) break;
      std::memcpy(host + c * chunk, slots + s * kRingSlot, size(c));
      if (c + 2 * nw < nchunks) issue(c + 2 * nw, s);
    }
  } else {
    for (size_t c = w; c < nchunks && e == hipSuccess; c += nw, s ^= 1) {
      if (c >= (size_t)w + 2 * nw) e = hipEventSynchronize(ev[s]);
      if (e != hipSuccess) break;
      std::memcpy(slots + s * kRingSlot, host + c * chunk, size(c));
      issue(c, s);
    }
  }
  for (auto& x : ev)
    if (x) {
      const hipError_t f = hipEventSynchronize(x);
      if (e == hipSuccess) e = f;
      (void)hipEventDestroy(x);
    }
  return e;
}

// Whether the runtime knows an address: pinned, managed or device memory, where its copy is one transfer
// without a staging buffer (256^3 from and to a pinned array 2.8 and 2.5 ms, through the ring 4.0 and 3.5).
inline bool ring_known(const void* p) {
  hipPointerAttribute_t a;
  if (hipPointerGetAttributes(&a, p) == hipSuccess) return a.type != hipMemoryTypeUnregistered;
  (void)hipGetLastError();  // an ordinary array
  return false;
}

// bytes between device and host memory behind the work on st; returns when done.
inline hipError_t ring_copy(int device, hipStream_t st, void* dev, void* host, size_t bytes, bool to_host) {
  std::unique_lock<std::mutex> lk(g_ring.use, std::defer_lock);
  if (bytes >= (to_host ? kRingToHost : kRingToDevice) && !ring_known(host) && lk.try_lock() && !g_ring.buf &&
      hipHostMalloc((void**)&g_ring.buf, kRingSlot * kRingSlots, hipHostMallocPortable) != hipSuccess) {
    (void)hipGetLastError();
    g_ring.buf = nullptr;
  }
  if (!lk.owns_lock() || !g_ring.buf) {
    const hipError_t e = to_host ? hipMemcpyAsync(host, dev, bytes, hipMemcpyDeviceToHost, st)
                                 : hipMemcpyAsync(dev, host, bytes, hipMemcpyHostToDevice, st);
    if (e != hipSuccess) return e;
    return hipStreamSynchronize(st);  // the host array is borrowed for the duration of the call only
  }
  // Worker threads meet the caller's own (an OpenMP team that still spins behind its last loop): 96^3 and
  // 128^3 into fresh arrays take 0.38 and 0.9-1.2 ms with one worker, 0.48 and 0.9-1.5 with four, so that
  // each further one has 32 MB to move.
  const size_t chunk = std::min(kRingSlot, (bytes / 8 + 4095) & ~(size_t)4095);
  const int nw = (int)std::min<size_t>(kRingWorkers, 1 + bytes / (16 * kRingSlot));
  std::atomic<int> err{hipSuccess};
  auto work = [&](int w) {
    const hipError_t e = ring_worker(device, st, (char*)dev, (char*)host, bytes, chunk, to_host, w, nw,
                                     g_ring.buf + 2 * kRingSlot * w);
    if (e != hipSuccess) err = e;
  };
  std::vector<std::thread> threads;
  int started = 0;
  try {
    threads.reserve(kRingWorkers);
    for (; started < nw - 1; ++started) threads.emplace_back(work, started + 1);
  } catch (const std::exception&) {  // no memory or no thread: this thread takes the rest
  }
  work(0);
  for (int w = started + 1; w < nw; ++w) work(w);  // those that could not be started
  for (auto& t : threads) t.join();
  // nothing may still use the slots or the caller's array when this returns, nor a copy whose event could not
  // be recorded
  const hipError_t e = hipStreamSynchronize(st);
  return err.load() != hipSuccess ? (hipError_t)err.load() : e;
}

}  // namespace smx
