// The pinned ring (smx_ring.h) over a stand-in for the runtime: copies are queued and made when something
// waits for them, and calls fail where they are told to.  Usage: ring_check <scenario>.
#include <cstdio>
#include <cstdlib>
#include <string>

#include "../smectic3d_amd/csrc/smx_ring.h"

namespace {
struct Op {
  void* dst;
  const void* src;
  size_t n;
};
std::mutex mu;
std::vector<Op> ops;     // in stream order
size_t done = 0;         // how many have been made
int copies = 0, records = 0, creates = 0, mallocs = 0;
int fail_record = -1, fail_copy = -1, fail_create = -1;  // the call that fails
bool fail_malloc = false;
hipMemoryType host_type = hipMemoryTypeUnregistered;
struct Ev { size_t at = 0; };
void run_to(size_t n) {
  for (; done < n; ++done) std::memcpy(ops[done].dst, ops[done].src, ops[done].n);
}
}  // namespace

extern "C" {
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetLastError() { return hipSuccess; }
hipError_t hipHostMalloc(void** p, size_t n, unsigned int) {
  ++mallocs;
  if (fail_malloc) return hipErrorOutOfMemory;
  *p = std::malloc(n);
  return hipSuccess;
}
hipError_t hipHostFree(void* p) {
  std::free(p);
  return hipSuccess;
}
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) {
  std::lock_guard<std::mutex> lk(mu);
  if (creates++ == fail_create) return hipErrorOutOfMemory;
  *e = reinterpret_cast<hipEvent_t>(new Ev());
  return hipSuccess;
}
hipError_t hipEventDestroy(hipEvent_t e) {
  delete reinterpret_cast<Ev*>(e);
  return hipSuccess;
}
hipError_t hipEventRecord(hipEvent_t e, hipStream_t) {
  std::lock_guard<std::mutex> lk(mu);
  if (records++ == fail_record) return hipErrorUnknown;
  reinterpret_cast<Ev*>(e)->at = ops.size();
  return hipSuccess;
}
hipError_t hipEventSynchronize(hipEvent_t e) {
  std::lock_guard<std::mutex> lk(mu);
  run_to(reinterpret_cast<Ev*>(e)->at);
  return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t) {
  std::lock_guard<std::mutex> lk(mu);
  run_to(ops.size());
  return hipSuccess;
}
hipError_t hipMemcpyAsync(void* dst, const void* src, size_t n, hipMemcpyKind, hipStream_t) {
  std::lock_guard<std::mutex> lk(mu);
  if (copies++ == fail_copy) return hipErrorUnknown;
  ops.push_back(Op{dst, src, n});
  return hipSuccess;
}
hipError_t hipPointerGetAttributes(hipPointerAttribute_t* a, const void*) {
  *a = hipPointerAttribute_t{};
  a->type = host_type;
  return hipSuccess;
}
}

static int bad(const char* what, size_t n, int k) {
  std::printf("FAILED: %s (%zu bytes, %d)\n", what, n, k);
  return 1;
}

// One transfer of n bytes; 0 where it returned `want` and, when that is success, moved every byte.
static int transfer(size_t n, bool to_host, hipError_t want, int k) {
  std::vector<char> dev(n), host(n);
  for (size_t i = 0; i < n; ++i) (to_host ? dev : host)[i] = (char)(i * 131 + (i >> 12) + 7);
  ops.clear();
  done = 0;
  copies = records = creates = 0;
  const hipError_t e = smx::ring_copy(0, nullptr, dev.data(), host.data(), n, to_host);
  if (done != ops.size()) return bad("copies still in flight on return", n, k);
  if ((e == hipSuccess) != (want == hipSuccess)) return bad("status", n, k);
  if (e == hipSuccess && std::memcmp(dev.data(), host.data(), n) != 0) return bad("bytes", n, k);
  return 0;
}

int main(int, char** argv) {
  const std::string what = argv[1];
  const size_t sizes[] = {4096, (4u << 20) - 8, 4u << 20, (4u << 20) + 8, (32u << 20) - 8, (32u << 20) + 24, 70000008};
  smx::ring_retain();
  int rc = 0;
  for (bool to_host : {true, false}) {
    if (what == "bytes") {
      for (size_t n : sizes) rc |= transfer(n, to_host, hipSuccess, 0);
    } else if (what == "errors") {
      for (size_t n : {(size_t)(33u << 20), (size_t)70000008}) {
        rc |= transfer(n, to_host, hipSuccess, 0);
        const int last = records - 1;  // behind the last copy of all
        for (int* f : {&fail_record, &fail_copy, &fail_create})
          for (int k : {0, 1, 2, 3, 7, last}) {
            if (f == &fail_create && k > 1) continue;
            *f = k;
            rc |= transfer(n, to_host, hipErrorUnknown, k);
            *f = -1;
            rc |= transfer(n, to_host, hipSuccess, k);  // the ring is free again
          }
      }
    } else if (what == "known") {
      for (hipMemoryType t : {hipMemoryTypeHost, hipMemoryTypeDevice, hipMemoryTypeManaged}) {
        host_type = t;
        rc |= transfer(70000008, to_host, hipSuccess, (int)t);
        if (copies != 1 || mallocs != 0) rc |= bad("not one copy of the runtime", 70000008, copies);
      }
    } else if (what == "nomemory") {
      fail_malloc = true;
      rc |= transfer(70000008, to_host, hipSuccess, 0);
    } else {
      return bad("no such scenario", 0, 0);
    }
  }
  smx::ring_release();
  if (what == "bytes" && smx::g_ring.buf) rc |= bad("ring kept after the last handle", 0, 0);
  if (rc == 0) std::printf("ok\n");
  return rc;
}
