/* Stand-ins for the HIP calls of csrc/transfer.cpp: copies are carried out when
 * something waits for them, and any call can be made to fail.  Test-only. */
#pragma once
#include <hip/hip_runtime.h>

#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <deque>
#include <map>
#include <mutex>

namespace fake {

struct Copy {
  void* dst;
  const void* src;
  size_t n;
};
inline std::mutex mu;
inline std::deque<Copy> pending;      // one queue for every stream
inline size_t done = 0;               // copies carried out
inline std::map<hipEvent_t, size_t> marks;
inline int records_left = -1;         // hipEventRecord calls until one fails; -1: none does
inline int host_allocations = 0, live_buffers = 0;
inline std::map<const void*, hipMemoryType> known;  // registered with the runtime

inline void run(size_t upto) {
  while (done < upto && !pending.empty()) {
    memcpy(pending.front().dst, pending.front().src, pending.front().n);
    pending.pop_front();
    done++;
  }
}

}  // namespace fake

extern "C" {
hipError_t hipHostMalloc(void** p, size_t n, unsigned int) {
  std::lock_guard<std::mutex> lk(fake::mu);
  fake::host_allocations++;
  fake::live_buffers++;
  *p = malloc(n);
  return hipSuccess;
}
hipError_t hipHostFree(void* p) {
  std::lock_guard<std::mutex> lk(fake::mu);
  fake::live_buffers--;
  free(p);
  return hipSuccess;
}
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) {
  *e = (hipEvent_t)malloc(1);
  return hipSuccess;
}
hipError_t hipEventDestroy(hipEvent_t e) {
  free((void*)e);
  return hipSuccess;
}
hipError_t hipEventRecord(hipEvent_t e, hipStream_t) {
  std::lock_guard<std::mutex> lk(fake::mu);
  if (fake::records_left >= 0 && fake::records_left-- == 0) return hipErrorInvalidHandle;
  fake::marks[e] = fake::done + fake::pending.size();
  return hipSuccess;
}
hipError_t hipEventSynchronize(hipEvent_t e) {
  std::lock_guard<std::mutex> lk(fake::mu);
  fake::run(fake::marks[e]);
  return hipSuccess;
}
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind, hipStream_t) {
  std::lock_guard<std::mutex> lk(fake::mu);
  fake::pending.push_back({d, s, n});
  return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t) {
  std::lock_guard<std::mutex> lk(fake::mu);
  fake::run(fake::done + fake::pending.size());
  return hipSuccess;
}
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetLastError(void) { return hipSuccess; }
hipError_t hipStreamCreate(hipStream_t* s) {
  *s = (hipStream_t)malloc(1);
  return hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t s) {
  free((void*)s);
  return hipSuccess;
}
hipError_t hipPointerGetAttributes(hipPointerAttribute_t* a, const void* p) {
  std::lock_guard<std::mutex> lk(fake::mu);
  memset(a, 0, sizeof *a);
  auto it = fake::known.find(p);
  a->type = it == fake::known.end() ? hipMemoryTypeUnregistered : it->second;
  return hipSuccess;
}
}
