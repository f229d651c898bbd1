// qs_pool.hip -- device memory and per-object workspaces kept between
// objects (interface in qs_internal.h).
//
// A register or an adjoint pass lives for one run of a program that makes
// the next one at once.  hipMalloc and hipFree of its buffers cost set-up
// time on every run, and the driver clears memory that is handed back before
// it gives it out again, at some 50 GB/s: an adjoint loop that allocated 6 GiB
// per 33 ms pass stalled now and then for 0.1 to 2 s, and a loop over 32 GiB
// registers took 0.96 s per pass of 0.38 s of work.  So freed blocks are kept,
// by size, and handed to the next caller of the same size.
//
// Bounds: all kept blocks together take at most an eighth of the device's
// memory, the oldest leave first; a block that has lain here for a second is
// given back, whatever goes on with the others, as long as more than
// kIdleKept bytes are kept; and when an allocation of this library fails,
// everything kept on the device is given back before it is tried again.  A
// program that needs the memory for something else at once calls
// qs_release_memory.  A block is handed in only when no GPU work uses it any
// more (its owner has drained its stream), so any thread and any stream may
// take it next.  Contents are whatever was there.
#include <hip/hip_runtime.h>

#include <chrono>
#include <condition_variable>
#include <cstdlib>
#include <iterator>
#include <list>
#include <mutex>
#include <new>
#include <system_error>
#include <thread>
#include <vector>

#include "qs_internal.h"

namespace qs {
namespace {

constexpr size_t kIdleKept = 64ull << 20;
constexpr auto kIdle = std::chrono::seconds(1);
constexpr size_t kMaxSpaces = 4;  // kept workspaces per device
constexpr int kMaxDevices = 64;   // memory of further ones is not kept

using Clock = std::chrono::steady_clock;

struct Block {
  void *p;
  size_t bytes;
  int device;
  Clock::time_point since;  // when it was handed in
};

struct Pool {
  std::mutex mu;
  std::list<Block> blocks;  // oldest first
  size_t kept = 0;          // bytes in blocks
  std::vector<Workspace *> spaces;
  size_t bound[kMaxDevices] = {};  // bytes kept per device at most, 0: not asked yet
  std::condition_variable wake;  // of the thread that gives back what is idle
  int freeing = 0;               // threads that are giving blocks back
  std::condition_variable freed;
  bool started = false, exits = false, stopping = false;
  Pool() { spaces.reserve(kMaxSpaces * kMaxDevices); }  // putting one back throws nothing
};

// Never destroyed: threads may free their registers while the process exits.
Pool &pool() {
  static Pool *p = new Pool();
  return *p;
}

// Take kept blocks of `device` (all devices: -1) that were handed in by
// `until` out, oldest first, until at most `keep` bytes are left there.  The
// caller frees them without the lock.
std::list<Block> take_out(Pool &p, int device, size_t keep,
                          Clock::time_point until = Clock::time_point::max()) {
  size_t kept = 0;
  for (const Block &b : p.blocks)
    if (device < 0 || b.device == device) kept += b.bytes;
  std::list<Block> out;
  for (auto it = p.blocks.begin(); it != p.blocks.end() && kept > keep && it->since <= until;) {
    if (device >= 0 && it->device != device) {
      ++it;
      continue;
    }
    const auto next = std::next(it);
    kept -= it->bytes;
    p.kept -= it->bytes;
    out.splice(out.end(), p.blocks, it);
    it = next;
  }
  return out;
}

// Free blocks that were taken out, without the lock; `freeing` counts the
// threads that do, so that a failed allocation can wait for them.
//
// Another thread may be recording a stream into a graph, in the mode that
// refuses every thread's frees (and breaks the recording off); these are none
// of the recorded work's.
void give_back(Pool &p, std::unique_lock<std::mutex> &lk, const std::list<Block> &v) {
  if (v.empty()) return;
  ++p.freeing;
  lk.unlock();
  hipStreamCaptureMode mode = hipStreamCaptureModeRelaxed;
  (void)hipThreadExchangeStreamCaptureMode(&mode);
  for (const Block &b : v) (void)hipFree(b.p);
  (void)hipThreadExchangeStreamCaptureMode(&mode);
  lk.lock();
  --p.freeing;
  p.freed.notify_all();
}

// Makes `device` current for a block of code.
struct OnDevice {
  int before = 0;
  bool moved = false;
  hipError_t error;
  explicit OnDevice(int device) {
    error = hipGetDevice(&before);
    if (error != hipSuccess || before == device) return;
    error = hipSetDevice(device);
    moved = error == hipSuccess;
  }
  ~OnDevice() {
    if (moved) (void)hipSetDevice(before);
  }
  OnDevice(const OnDevice &) = delete;
  OnDevice &operator=(const OnDevice &) = delete;
};

bool out_of_memory(hipError_t e) {
  return e == hipErrorOutOfMemory || e == hipErrorMemoryAllocation;
}

void idle_thread() {
  Pool &p = pool();
  std::unique_lock<std::mutex> lk(p.mu);
  while (!p.stopping) {
    if (p.kept <= kIdleKept) {
      p.wake.wait(lk);
      continue;
    }
    const auto now = Clock::now();
    const auto due = p.blocks.front().since + kIdle;
    if (now < due) {
      p.wake.wait_until(lk, due);
      continue;
    }
    give_back(p, lk, take_out(p, -1, kIdleKept, now - kIdle));
  }
}

// At exit (before the runtime is torn down): no frees from here on, and none
// under way.
void stop_idle_thread() {
  Pool &p = pool();
  std::unique_lock<std::mutex> lk(p.mu);
  p.stopping = true;
  p.freed.wait(lk, [&] { return p.freeing == 0; });
}

// Whether the idle thread runs (it is started on demand): without it nothing
// would be given back, so nothing above kIdleKept is kept.
bool idle_thread_runs(Pool &p) {
  if (p.started) return true;
  if (p.exits || std::atexit(stop_idle_thread) == 0) {
    p.exits = true;
    try {
      std::thread(idle_thread).detach();
      p.started = true;
    } catch (const std::system_error &) {
    }
  }
  return p.started;
}

}  // namespace

hipError_t pool_malloc(void **out, size_t bytes, int device) {
  *out = nullptr;
  Pool &p = pool();
  {
    std::lock_guard<std::mutex> lk(p.mu);
    for (auto it = p.blocks.end(); it != p.blocks.begin();) {
      --it;  // the newest first
      if (it->bytes == bytes && it->device == device) {
        *out = it->p;
        p.kept -= bytes;
        p.blocks.erase(it);
        return hipSuccess;
      }
    }
  }
  const OnDevice on(device);
  if (on.error != hipSuccess) return on.error;
  const hipError_t e = hipMalloc(out, bytes);
  if (!out_of_memory(e)) return e;
  (void)hipGetLastError();
  std::unique_lock<std::mutex> lk(p.mu);
  give_back(p, lk, take_out(p, device, 0));
  // (also when nothing was kept: another thread may just be giving it back)
  p.freed.wait(lk, [&] { return p.freeing == 0; });
  lk.unlock();
  return hipMalloc(out, bytes);
}

// No exception leaves it: closing a register ends here, at a C entry.
void pool_free(void *ptr, size_t bytes, int device) {
  if (!ptr) return;
  Pool &p = pool();
  std::list<Block> freed;
  try {
    freed.push_back({ptr, bytes, device, Clock::now()});
  } catch (const std::bad_alloc &) {
    (void)hipFree(ptr);
    return;
  }
  std::unique_lock<std::mutex> lk(p.mu);
  if (bytes > 0 && device >= 0 && device < kMaxDevices) {
    size_t &bound = p.bound[device];  // bytes kept there at most
    if (bound == 0) {
      size_t total = 0;
      hipDevice_t d = 0;
      if (hipDeviceGet(&d, device) == hipSuccess && hipDeviceTotalMem(&total, d) == hipSuccess)
        bound = total / 8;
    }
    if (bytes <= bound && !p.stopping) {
      p.kept += bytes;
      p.blocks.splice(p.blocks.end(), freed);
      freed = take_out(p, device, bound);
      if (p.kept > kIdleKept && !idle_thread_runs(p))
        freed.splice(freed.end(), take_out(p, -1, kIdleKept));
      p.wake.notify_one();
    }
  }
  give_back(p, lk, freed);
}

namespace {

void destroy(Workspace *w) {
  pool_free(w->d_ring, kRingBytes, w->device);
  if (w->h_ring) (void)hipHostFree(w->h_ring);
  pool_free(w->d_red, kRedDoubles * sizeof(double), w->device);
  if (w->h_red) (void)hipHostFree(w->h_red);
  if (w->stream) (void)hipStreamDestroy(w->stream);
  delete w;
}

}  // namespace

hipError_t workspace_get(Workspace **out, int device) {
  *out = nullptr;
  Pool &p = pool();
  {
    std::lock_guard<std::mutex> lk(p.mu);
    for (size_t i = p.spaces.size(); i-- > 0;)
      if (p.spaces[i]->device == device) {
        *out = p.spaces[i];
        p.spaces.erase(p.spaces.begin() + (long)i);
        return hipSuccess;
      }
  }
  Workspace *w = new Workspace();
  w->device = device;
  const OnDevice on(device);
  hipError_t e = on.error;
  if (e == hipSuccess) e = hipStreamCreateWithFlags(&w->stream, hipStreamNonBlocking);
  if (e == hipSuccess) e = pool_malloc((void **)&w->d_red, kRedDoubles * sizeof(double), device);
  if (e == hipSuccess) e = hipHostMalloc((void **)&w->h_red, 64 * sizeof(double));
  if (e == hipSuccess) e = pool_malloc((void **)&w->d_ring, kRingBytes, device);
  if (e == hipSuccess) e = hipHostMalloc((void **)&w->h_ring, kRingBytes);
  // measurement slots that nothing has written read 0
  if (e == hipSuccess)
    e = hipMemsetAsync(w->d_red, 0, kRedDoubles * sizeof(double), w->stream);
  if (e != hipSuccess) {
    destroy(w);
    return e;
  }
  *out = w;
  return hipSuccess;
}

void workspace_put(Workspace *w) {
  if (!w) return;
  Pool &p = pool();
  {
    std::lock_guard<std::mutex> lk(p.mu);
    size_t n = 0;
    for (const Workspace *s : p.spaces) n += s->device == w->device;
    if (n < kMaxSpaces && p.spaces.size() < p.spaces.capacity()) {
      p.spaces.push_back(w);
      return;
    }
  }
  destroy(w);
}

void pool_release() {
  Pool &p = pool();
  std::unique_lock<std::mutex> lk(p.mu);
  while (!p.spaces.empty()) {
    Workspace *w = p.spaces.back();
    p.spaces.pop_back();
    lk.unlock();
    destroy(w);
    lk.lock();
  }
  give_back(p, lk, take_out(p, -1, 0));
  p.freed.wait(lk, [&] { return p.freeing == 0; });
}

}  // namespace qs
