// fake_hip.hpp -- the HIP runtime calls of libsgtsne_hip.so, defined in a test
// program that links it: kernels do nothing, device memory is only counted, and
// any call can be made to fail.  The library's host code (allocation, release,
// error paths) then runs without a GPU.
//
// Device memory has a capacity.  Stream-ordered frees go to the stream's share of
// the pool; another stream gets that memory only once the freeing stream has been
// synchronised and the pool trimmed, or after waiting for an event recorded there:
// the rules this library sets for the pool.
#pragma once
#ifndef __HIP_PLATFORM_AMD__
#define __HIP_PLATFORM_AMD__
#endif
#include <hip/hip_runtime_api.h>

#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <set>
#include <string>

namespace fake {

struct Block {
  size_t bytes;
  bool pooled;  // allocated from the pool
};
inline std::map<uintptr_t, Block> live;
inline std::map<uintptr_t, size_t> pool;  // stream -> bytes freed there
inline std::set<uintptr_t> busy;          // streams with frees since their last synchronisation
inline size_t capacity = ~(size_t)0 >> 2;
inline uintptr_t next_address = (uintptr_t)1 << 40;
inline hipError_t last = hipSuccess;

inline std::string fail_call;  // the call that fails ...
inline long fail_from = -1;    // ... from its fail_from-th use on (counted from 0)
inline std::map<std::string, long> calls;

inline void reset_calls() { calls.clear(); }
inline void fail(const char *call, long from) {
  calls.clear();
  fail_call = call;
  fail_from = from;
}
inline void succeed() { fail_call.clear(); }
inline bool failing(const char *call) { return calls[call]++ >= fail_from && fail_call == call; }

inline size_t live_bytes() {
  size_t b = 0;
  for (auto &e : live) b += e.second.bytes;
  return b;
}
inline size_t pool_bytes() {
  size_t b = 0;
  for (auto &e : pool) b += e.second;
  return b;
}

inline hipError_t alloc(void **p, size_t bytes, bool pooled, uintptr_t s) {
  if (pooled) {
    const size_t mine = pool[s] < bytes ? pool[s] : bytes;
    if (bytes - mine > capacity - live_bytes() - pool_bytes()) return last = hipErrorOutOfMemory;
    pool[s] -= mine;
  } else if (bytes > capacity - live_bytes() - pool_bytes()) {
    return last = hipErrorOutOfMemory;
  }
  *p = reinterpret_cast<void *>(next_address);
  live[next_address] = Block{bytes, pooled};
  next_address += (bytes + 4095) / 4096 * 4096 + 4096;
  return hipSuccess;
}

}  // namespace fake

#define FAKE_FAIL(name, code) \
  if (fake::failing(#name)) return fake::last = code

extern "C" {

void **__hipRegisterFatBinary(const void *) {
  static void *handle = nullptr;
  return &handle;
}
void __hipUnregisterFatBinary(void **) {}
void __hipRegisterFunction(void **, const void *, char *, const char *, unsigned, void *, void *, void *, void *, int *) {}
void __hipRegisterVar(void **, void *, char *, char *, int, size_t, int, int) {}
hipError_t __hipPushCallConfiguration(dim3, dim3, size_t, hipStream_t) { return hipSuccess; }
hipError_t __hipPopCallConfiguration(dim3 *, dim3 *, size_t *, hipStream_t *) { return hipSuccess; }

hipError_t hipLaunchKernel(const void *, dim3, dim3, void **, size_t, hipStream_t) {
  FAKE_FAIL(hipLaunchKernel, hipErrorLaunchFailure);
  return hipSuccess;
}
hipError_t hipGetLastError(void) {
  const hipError_t e = fake::last;
  fake::last = hipSuccess;
  return e;
}
const char *hipGetErrorString(hipError_t) { return "fake"; }
hipError_t hipGetDeviceCount(int *n) {
  *n = 1;
  return hipSuccess;
}
hipError_t hipGetDevice(int *d) {
  *d = 0;
  return hipSuccess;
}
hipError_t hipDeviceGetAttribute(int *v, hipDeviceAttribute_t, int) {
  *v = 100000;
  return hipSuccess;
}
hipError_t hipGetDevicePropertiesR0600(hipDeviceProp_tR0600 *p, int) {
  std::memset(p, 0, sizeof(*p));
  std::strcpy(p->gcnArchName, "gfx950");
  p->multiProcessorCount = 256;
  p->warpSize = 64;
  p->maxThreadsPerBlock = 1024;
  p->maxGridSize[0] = 2147483647;
  p->sharedMemPerBlock = 65536;
  return hipSuccess;
}
int hipGetStreamDeviceId(hipStream_t) { return 0; }
hipError_t hipGetSymbolAddress(void **p, const void *) {
  *p = reinterpret_cast<void *>(fake::next_address);
  return hipSuccess;
}

hipError_t hipMalloc(void **p, size_t n) {
  FAKE_FAIL(hipMalloc, hipErrorOutOfMemory);
  return fake::alloc(p, n, false, 0);
}
hipError_t hipFree(void *p) {
  if (p && !fake::live.erase(reinterpret_cast<uintptr_t>(p))) std::abort();  // freed twice
  return hipSuccess;
}
hipError_t hipMallocAsync(void **p, size_t n, hipStream_t s) {
  FAKE_FAIL(hipMallocAsync, hipErrorOutOfMemory);
  return fake::alloc(p, n, true, reinterpret_cast<uintptr_t>(s));
}
hipError_t hipFreeAsync(void *p, hipStream_t s) {
  if (!p) return hipSuccess;
  auto it = fake::live.find(reinterpret_cast<uintptr_t>(p));
  if (it == fake::live.end() || !it->second.pooled) std::abort();
  fake::pool[reinterpret_cast<uintptr_t>(s)] += it->second.bytes;
  fake::busy.insert(reinterpret_cast<uintptr_t>(s));
  fake::live.erase(it);
  return hipSuccess;
}
hipError_t hipDeviceGetDefaultMemPool(hipMemPool_t *p, int) {
  *p = reinterpret_cast<hipMemPool_t>(1);
  return hipSuccess;
}
hipError_t hipMemPoolSetAttribute(hipMemPool_t, hipMemPoolAttr, void *) { return hipSuccess; }
hipError_t hipMemPoolTrimTo(hipMemPool_t, size_t) {
  for (auto &e : fake::pool)
    if (!fake::busy.count(e.first)) e.second = 0;
  return hipSuccess;
}
hipError_t hipHostMalloc(void **p, size_t n, unsigned) {
  FAKE_FAIL(hipHostMalloc, hipErrorOutOfMemory);
  *p = std::calloc(1, n);
  return hipSuccess;
}
hipError_t hipHostFree(void *p) {
  std::free(p);
  return hipSuccess;
}

// device -> host copies deliver zeros, the others nothing
static hipError_t fake_copy(void *dst, size_t n, hipMemcpyKind kind) {
  if (kind == hipMemcpyDeviceToHost) std::memset(dst, 0, n);
  return hipSuccess;
}
hipError_t hipMemcpy(void *dst, const void *, size_t n, hipMemcpyKind kind) { return fake_copy(dst, n, kind); }
hipError_t hipMemcpyAsync(void *dst, const void *, size_t n, hipMemcpyKind kind, hipStream_t) {
  FAKE_FAIL(hipMemcpyAsync, hipErrorUnknown);
  return fake_copy(dst, n, kind);
}
hipError_t hipMemcpyWithStream(void *dst, const void *, size_t n, hipMemcpyKind kind, hipStream_t) {
  return fake_copy(dst, n, kind);
}
hipError_t hipMemset(void *, int, size_t) { return hipSuccess; }
hipError_t hipMemsetAsync(void *, int, size_t, hipStream_t) { return hipSuccess; }

hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned) {
  *s = reinterpret_cast<hipStream_t>(std::malloc(16));
  return hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t s) {
  std::free(reinterpret_cast<void *>(s));
  return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t s) {
  FAKE_FAIL(hipStreamSynchronize, hipErrorUnknown);
  fake::busy.erase(reinterpret_cast<uintptr_t>(s));
  return hipSuccess;
}
hipError_t hipStreamQuery(hipStream_t) { return hipSuccess; }

struct FakeEvent {
  uintptr_t stream;
};
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) {
  FAKE_FAIL(hipEventCreateWithFlags, hipErrorUnknown);
  *e = reinterpret_cast<hipEvent_t>(new FakeEvent{0});
  return hipSuccess;
}
hipError_t hipEventCreate(hipEvent_t *e) { return hipEventCreateWithFlags(e, 0); }
hipError_t hipEventDestroy(hipEvent_t e) {
  delete reinterpret_cast<FakeEvent *>(e);
  return hipSuccess;
}
hipError_t hipEventRecord(hipEvent_t e, hipStream_t s) {
  FAKE_FAIL(hipEventRecord, hipErrorUnknown);
  reinterpret_cast<FakeEvent *>(e)->stream = reinterpret_cast<uintptr_t>(s);
  return hipSuccess;
}
hipError_t hipEventQuery(hipEvent_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float *t, hipEvent_t, hipEvent_t) {
  *t = 1.0f;
  return hipSuccess;
}
hipError_t hipStreamWaitEvent(hipStream_t s, hipEvent_t e, unsigned) {
  const uintptr_t from = reinterpret_cast<FakeEvent *>(e)->stream, to = reinterpret_cast<uintptr_t>(s);
  if (from != to) {
    fake::pool[to] += fake::pool[from];
    fake::pool[from] = 0;
  }
  return hipSuccess;
}

hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) { return hipSuccess; }
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t *g) {
  *g = reinterpret_cast<hipGraph_t>(1);
  return hipSuccess;
}
hipError_t hipGraphInstantiate(hipGraphExec_t *e, hipGraph_t, hipGraphNode_t *, char *, size_t) {
  *e = reinterpret_cast<hipGraphExec_t>(1);
  return hipSuccess;
}
hipError_t hipGraphExecUpdate(hipGraphExec_t, hipGraph_t, hipGraphNode_t *, hipGraphExecUpdateResult *r) {
  *r = hipGraphExecUpdateSuccess;
  return hipSuccess;
}
hipError_t hipGraphLaunch(hipGraphExec_t, hipStream_t) { return hipSuccess; }
hipError_t hipGraphDestroy(hipGraph_t) { return hipSuccess; }
hipError_t hipGraphExecDestroy(hipGraphExec_t) { return hipSuccess; }

}  // extern "C"

#define EXPECT(cond)                                                   \
  do {                                                                 \
    if (!(cond)) {                                                     \
      std::printf("%s:%d: %s\n", __FILE__, __LINE__, #cond);           \
      return 1;                                                        \
    }                                                                  \
  } while (0)
