// Staged copies between pageable host memory and the device.
//
// hipMemcpy on pageable memory pins and unpins the caller's pages or stages
// them on one thread: 1 MB takes 380-450 us either way where pinned memory
// takes 27, and 75 MB down to a fresh array 7.6 ms where the DMA takes 1.4.
// Here up to eight threads each move a slice through two pinned buffers of 1
// MB, so that the host-side copies and the page faults of a fresh array run in
// parallel and overlap the DMA: weno_solver's 8 MB up and 75 MB
// down, whole call, 29.5 -> 4.0 ms (with the rows formed on the device), ten
// steps of a 2048 x 2048 grid with its state up and down 55.5 -> 46.6 ms.
#include "transfer.h"

#include <algorithm>
#include <cstring>
#include <mutex>
#include <system_error>
#include <thread>
#include <vector>

namespace pypde {
namespace {

constexpr size_t CHUNK = 1u << 20;
constexpr int MAX_LANES = 8;  // per copy, and kept idle per process (16 MB pinned)

struct Lane {
  int device = -1;
  void* buf[2] = {nullptr, nullptr};
  hipEvent_t ev[2] = {nullptr, nullptr};
};

std::mutex g_mu;
std::vector<Lane*> g_lanes;                            // idle
std::vector<std::pair<int, hipStream_t>> g_streams;    // idle

void destroy(Lane* l) {
  for (int i = 0; i < 2; i++) {
    if (l->ev[i]) (void)hipEventDestroy(l->ev[i]);
    if (l->buf[i]) (void)hipHostFree(l->buf[i]);
  }
  delete l;
}

Lane* take_lane(int device) {
  {
    std::lock_guard<std::mutex> lk(g_mu);
    for (size_t i = 0; i < g_lanes.size(); i++)
      if (g_lanes[i]->device == device) {
        Lane* l = g_lanes[i];
        g_lanes.erase(g_lanes.begin() + (long)i);
        return l;
      }
  }
  Lane* l = new Lane();
  l->device = device;
  for (int i = 0; i < 2; i++)
    if (hipHostMalloc(&l->buf[i], CHUNK, hipHostMallocDefault) != hipSuccess ||
        hipEventCreateWithFlags(&l->ev[i], hipEventDisableTiming) != hipSuccess) {
      (void)hipGetLastError();
      destroy(l);
      return nullptr;
    }
  return l;
}

// Every copy through the lane has completed.
void give_lane(Lane* l) {
  {
    std::lock_guard<std::mutex> lk(g_mu);
    if (g_lanes.size() < (size_t)MAX_LANES) {
      g_lanes.push_back(l);
      return;
    }
  }
  destroy(l);
}

hipError_t slice_up(Lane* l, char* dev, const char* host, size_t n, hipStream_t s) {
  bool used[2] = {false, false};
  hipError_t e = hipSuccess;
  for (size_t off = 0, k = 0; off < n && e == hipSuccess; off += CHUNK, k ^= 1) {
    const size_t len = std::min(CHUNK, n - off);
    if (used[k]) e = hipEventSynchronize(l->ev[k]);
    if (e != hipSuccess) break;
    memcpy(l->buf[k], host + off, len);
    e = hipMemcpyAsync(dev + off, l->buf[k], len, hipMemcpyHostToDevice, s);
    if (e == hipSuccess) e = hipEventRecord(l->ev[k], s);
    used[k] = e == hipSuccess;
  }
  for (int k = 0; k < 2; k++)
    if (used[k]) {
      const hipError_t w = hipEventSynchronize(l->ev[k]);
      if (e == hipSuccess) e = w;
    }
  if (e != hipSuccess) (void)hipStreamSynchronize(s);  // nothing may still read the lane
  return e;
}

hipError_t slice_down(Lane* l, char* host, const char* dev, size_t n, hipStream_t s) {
  hipError_t e = hipSuccess;
  const size_t chunks = (n + CHUNK - 1) / CHUNK;
  auto len = [&](size_t c) { return std::min(CHUNK, n - c * CHUNK); };
  size_t queued = 0;
  for (size_t c = 0; c < chunks && e == hipSuccess; c++) {
    for (; queued < chunks && queued < c + 2 && e == hipSuccess; queued++) {
      e = hipMemcpyAsync(l->buf[queued & 1], dev + queued * CHUNK, len(queued),
                         hipMemcpyDeviceToHost, s);
      if (e == hipSuccess) e = hipEventRecord(l->ev[queued & 1], s);
    }
    if (e == hipSuccess) e = hipEventSynchronize(l->ev[c & 1]);
    if (e == hipSuccess) memcpy(host + c * CHUNK, l->buf[c & 1], len(c));
  }
  if (e != hipSuccess) (void)hipStreamSynchronize(s);  // nothing may still write the lane
  return e;
}

template <typename Slice>
hipError_t staged(size_t n, int device, Slice slice) {
  const int want = (int)std::min<size_t>(MAX_LANES, std::max<size_t>(1, n / CHUNK));
  std::vector<Lane*> lanes;
  while ((int)lanes.size() < want) {
    Lane* l = take_lane(device);
    if (!l) break;
    lanes.push_back(l);
  }
  if (lanes.empty()) return hipErrorOutOfMemory;
  const size_t T = lanes.size();
  const size_t per = ((n + T - 1) / T + 4095) / 4096 * 4096;
  std::vector<hipError_t> err(T, hipSuccess);
  auto work = [&](size_t t) {
    const size_t a = std::min(n, t * per), b = std::min(n, (t + 1) * per);
    if (a == b) return;
    if (t) err[t] = hipSetDevice(device);
    if (err[t] == hipSuccess) err[t] = slice(lanes[t], a, b - a);
  };
  std::vector<std::thread> th;
  size_t started = 1;
  try {
    for (; started < T; started++) th.emplace_back(work, started);
  } catch (const std::system_error&) {
    // no more threads: the rest runs here
  }
  work(0);
  for (size_t t = started; t < T; t++) work(t);
  for (auto& x : th) x.join();
  for (Lane* l : lanes) give_lane(l);
  for (hipError_t e : err)
    if (e != hipSuccess) return e;
  return hipSuccess;
}

// Pinned, managed and device memory, which the runtime copies by itself without
// staging (and the host may not be able to read).
bool known_to_runtime(const void* p) {
  hipPointerAttribute_t a;
  if (hipPointerGetAttributes(&a, p) == hipSuccess) return a.type != hipMemoryTypeUnregistered;
  (void)hipGetLastError();
  return false;
}

hipError_t direct(void* dst, const void* src, size_t n, hipMemcpyKind kind, hipStream_t s) {
  const hipError_t e = hipMemcpyAsync(dst, src, n, kind, s);
  return e == hipSuccess ? hipStreamSynchronize(s) : e;
}

}  // namespace

hipError_t copy_to_device(void* dev, const void* host, size_t n, int device, hipStream_t s) {
  if (!n) return hipSuccess;
  if (known_to_runtime(host)) return direct(dev, host, n, hipMemcpyDefault, s);
  const hipError_t e = staged(n, device, [&](Lane* l, size_t a, size_t len) {
    return slice_up(l, (char*)dev + a, (const char*)host + a, len, s);
  });
  return e == hipErrorOutOfMemory ? direct(dev, host, n, hipMemcpyHostToDevice, s) : e;
}

hipError_t copy_to_host(void* host, const void* dev, size_t n, int device, hipStream_t s) {
  if (!n) return hipSuccess;
  if (known_to_runtime(host)) return direct(host, dev, n, hipMemcpyDefault, s);
  const hipError_t e = staged(n, device, [&](Lane* l, size_t a, size_t len) {
    return slice_down(l, (char*)host + a, (const char*)dev + a, len, s);
  });
  return e == hipErrorOutOfMemory ? direct(host, dev, n, hipMemcpyDeviceToHost, s) : e;
}

hipError_t take_stream(int device, hipStream_t* s) {
  {
    std::lock_guard<std::mutex> lk(g_mu);
    for (size_t i = 0; i < g_streams.size(); i++)
      if (g_streams[i].first == device) {
        *s = g_streams[i].second;
        g_streams.erase(g_streams.begin() + (long)i);
        return hipSuccess;
      }
  }
  return hipStreamCreate(s);
}

void give_stream(int device, hipStream_t s) {
  {
    std::lock_guard<std::mutex> lk(g_mu);
    if (g_streams.size() < 8) {
      g_streams.push_back({device, s});
      return;
    }
  }
  (void)hipStreamDestroy(s);
}

void release_idle_transfer() {
  std::vector<Lane*> lanes;
  std::vector<std::pair<int, hipStream_t>> streams;
  {
    std::lock_guard<std::mutex> lk(g_mu);
    lanes.swap(g_lanes);
    streams.swap(g_streams);
  }
  for (Lane* l : lanes) destroy(l);
  for (auto& x : streams) (void)hipStreamDestroy(x.second);
}

}  // namespace pypde
