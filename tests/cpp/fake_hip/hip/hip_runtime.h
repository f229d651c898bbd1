// A stand-in for the HIP runtime on the CPU: two devices with a number of
// bytes each, and nothing behind the addresses.  It covers what qs_pool.hip
// calls, so that pool_check.cpp runs that file itself without a GPU.
#pragma once

#include <atomic>
#include <chrono>
#include <cstddef>
#include <cstdint>
#include <map>
#include <mutex>
#include <thread>

enum hipError_t {
  hipSuccess = 0,
  hipErrorInvalidValue = 1,
  hipErrorOutOfMemory = 2,
  hipErrorMemoryAllocation = hipErrorOutOfMemory,
  hipErrorInvalidDevice = 101,
  hipErrorStreamCaptureUnsupported = 900,
};
enum hipStreamCaptureMode {
  hipStreamCaptureModeGlobal = 0,
  hipStreamCaptureModeThreadLocal = 1,
  hipStreamCaptureModeRelaxed = 2,
};
typedef int hipDevice_t;
typedef struct fakeStream *hipStream_t;
constexpr unsigned hipStreamNonBlocking = 1;

namespace fake {

constexpr int kDevices = 2;

struct Runtime {
  std::mutex mu;
  size_t total[kDevices] = {64ull << 30, 64ull << 30}, used[kDevices] = {0, 0};
  std::map<void *, std::pair<int, size_t>> live;  // address: device, bytes
  uintptr_t next = 1ull << 20;
  size_t mallocs = 0, frees = 0, refused_frees = 0;
  bool capturing = false;  // some thread records a stream in the global mode
};

inline Runtime &rt() {
  static Runtime *r = new Runtime();
  return *r;
}

inline thread_local int current = 0;
inline thread_local hipStreamCaptureMode mode = hipStreamCaptureModeGlobal;
inline std::atomic<int> free_ms{0};  // how long a free waits for the device
inline std::atomic<int> streams{0}, host_blocks{0};

// Device of a live block, -1: none there.
inline int device_of(void *p) {
  std::lock_guard<std::mutex> lk(rt().mu);
  auto it = rt().live.find(p);
  return it == rt().live.end() ? -1 : it->second.first;
}

inline size_t used(int device) {
  std::lock_guard<std::mutex> lk(rt().mu);
  return rt().used[device];
}

}  // namespace fake

inline hipError_t hipGetDevice(int *d) {
  *d = fake::current;
  return hipSuccess;
}
inline hipError_t hipSetDevice(int d) {
  if (d < 0 || d >= fake::kDevices) return hipErrorInvalidDevice;
  fake::current = d;
  return hipSuccess;
}
inline hipError_t hipDeviceGet(hipDevice_t *out, int d) {
  *out = d;
  return d >= 0 && d < fake::kDevices ? hipSuccess : hipErrorInvalidDevice;
}
inline hipError_t hipDeviceTotalMem(size_t *out, hipDevice_t d) {
  *out = fake::rt().total[d];
  return hipSuccess;
}
inline hipError_t hipGetLastError() { return hipSuccess; }
inline hipError_t hipThreadExchangeStreamCaptureMode(hipStreamCaptureMode *m) {
  const hipStreamCaptureMode old = fake::mode;
  fake::mode = *m;
  *m = old;
  return hipSuccess;
}
inline hipError_t hipMalloc(void **out, size_t bytes) {
  auto &r = fake::rt();
  std::lock_guard<std::mutex> lk(r.mu);
  const int d = fake::current;
  ++r.mallocs;
  *out = nullptr;
  if (r.capturing && fake::mode != hipStreamCaptureModeRelaxed)
    return hipErrorStreamCaptureUnsupported;
  if (r.used[d] + bytes > r.total[d]) return hipErrorOutOfMemory;
  r.used[d] += bytes;
  *out = (void *)r.next;
  r.next += 1 << 20;
  r.live[*out] = {d, bytes};
  return hipSuccess;
}
inline hipError_t hipFree(void *p) {
  auto &r = fake::rt();
  std::this_thread::sleep_for(std::chrono::milliseconds(fake::free_ms.load()));
  std::lock_guard<std::mutex> lk(r.mu);
  if (r.capturing && fake::mode != hipStreamCaptureModeRelaxed) {
    ++r.refused_frees;
    return hipErrorStreamCaptureUnsupported;
  }
  auto it = r.live.find(p);
  if (it == r.live.end()) return hipErrorInvalidValue;
  ++r.frees;
  r.used[it->second.first] -= it->second.second;
  r.live.erase(it);
  return hipSuccess;
}
template <typename T>
hipError_t hipHostMalloc(T **out, size_t) {
  *out = reinterpret_cast<T *>(new char[16]);
  ++fake::host_blocks;
  return hipSuccess;
}
inline hipError_t hipHostFree(void *p) {
  delete[] static_cast<char *>(p);
  --fake::host_blocks;
  return hipSuccess;
}
inline hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned) {
  *s = reinterpret_cast<hipStream_t>(new char[1]);
  ++fake::streams;
  return hipSuccess;
}
inline hipError_t hipStreamDestroy(hipStream_t s) {
  delete[] reinterpret_cast<char *>(s);
  --fake::streams;
  return hipSuccess;
}
inline hipError_t hipMemsetAsync(void *, int, size_t, hipStream_t) { return hipSuccess; }
