// qs_pool.hip -- device memory and per-object workspaces kept between
// objects (interface in qs_internal.h).
//
// A register or an adjoint pass lives for one run of a program that makes
// the next one at once.  hipMalloc and hipFree of its buffers cost set-up
// time on every run, and memory handed back and taken again at many GB/s
// makes the driver clear it each time: an adjoint loop that allocated 6 GiB
// per 33 ms pass stalled now and then for 0.1 to 2 s.  So freed blocks are
// kept, by size, and handed to the next caller of the same size.
//
// Bounds: blocks of more than kMaxBlock bytes are never kept, all kept blocks
// together take at most kMaxKept bytes per device, the oldest leave first;
// when the last register and circuit is gone, all but kIdleKept bytes are
// given back; and when an allocation of this library fails, everything kept
// on the device is given back before it is tried again.  A block is handed
// in only when no GPU work uses it any more (its owner has drained its
// stream), so any thread and any stream may take it next.  Contents are
// whatever was there.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <list>
#include <mutex>
#include <vector>

#include "qs_internal.h"

namespace qs {
namespace {

constexpr size_t kMaxBlock = 2ull << 30;
constexpr size_t kMaxKept = 8ull << 30;
constexpr size_t kIdleKept = 64ull << 20;
constexpr size_t kMaxSpaces = 4;  // kept workspaces per device

struct Block {
  void *p;
  size_t bytes;
  int device;
};

struct Pool {
  std::mutex mu;
  std::list<Block> blocks;  // oldest first
  std::vector<Workspace *> spaces;
  size_t live = 0;  // registers and circuits
};

// Never destroyed: threads may free their registers while the process exits.
Pool &pool() {
  static Pool *p = new Pool();
  return *p;
}

// Take kept blocks of `device` (all devices: -1) out, oldest first, until at
// most `keep` bytes are left there.  The caller frees them without the lock.
std::vector<Block> take_out(Pool &p, int device, size_t keep) {
  size_t kept = 0;
  for (const Block &b : p.blocks)
    if (device < 0 || b.device == device) kept += b.bytes;
  std::vector<Block> out;
  for (auto it = p.blocks.begin(); it != p.blocks.end() && kept > keep;) {
    if (device >= 0 && it->device != device) {
      ++it;
      continue;
    }
    kept -= it->bytes;
    out.push_back(*it);
    it = p.blocks.erase(it);
  }
  return out;
}

void give_back(const std::vector<Block> &v) {
  for (const Block &b : v) (void)hipFree(b.p);
}

bool out_of_memory(hipError_t e) {
  return e == hipErrorOutOfMemory || e == hipErrorMemoryAllocation;
}

}  // namespace

hipError_t pool_malloc(void **out, size_t bytes) {
  *out = nullptr;
  int device = 0;
  hipError_t e = hipGetDevice(&device);
  if (e != hipSuccess) return e;
  Pool &p = pool();
  {
    std::lock_guard<std::mutex> lk(p.mu);
    for (auto it = p.blocks.end(); it != p.blocks.begin();) {
      --it;  // the newest first
      if (it->bytes == bytes && it->device == device) {
        *out = it->p;
        p.blocks.erase(it);
        return hipSuccess;
      }
    }
  }
  e = hipMalloc(out, bytes);
  if (!out_of_memory(e)) return e;
  std::vector<Block> freed;
  {
    std::lock_guard<std::mutex> lk(p.mu);
    freed = take_out(p, device, 0);
  }
  if (freed.empty()) return e;
  (void)hipGetLastError();
  give_back(freed);
  return hipMalloc(out, bytes);
}

void pool_free(void *ptr, size_t bytes, int device) {
  if (!ptr) return;
  if (bytes == 0 || bytes > kMaxBlock) {
    (void)hipFree(ptr);
    return;
  }
  Pool &p = pool();
  std::vector<Block> freed;
  {
    std::lock_guard<std::mutex> lk(p.mu);
    p.blocks.push_back({ptr, bytes, device});
    freed = take_out(p, device, kMaxKept);
  }
  give_back(freed);
}

void pool_retain() {
  Pool &p = pool();
  std::lock_guard<std::mutex> lk(p.mu);
  ++p.live;
}

void pool_release() {
  Pool &p = pool();
  std::vector<Block> freed;
  {
    std::lock_guard<std::mutex> lk(p.mu);
    if (--p.live == 0) freed = take_out(p, -1, kIdleKept);
  }
  give_back(freed);
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

hipError_t workspace_get(Workspace **out) {
  *out = nullptr;
  int device = 0;
  hipError_t e = hipGetDevice(&device);
  if (e != hipSuccess) return e;
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
  e = hipStreamCreateWithFlags(&w->stream, hipStreamNonBlocking);
  if (e == hipSuccess) e = pool_malloc((void **)&w->d_red, kRedDoubles * sizeof(double));
  if (e == hipSuccess) e = hipHostMalloc((void **)&w->h_red, 64 * sizeof(double));
  if (e == hipSuccess) e = pool_malloc((void **)&w->d_ring, kRingBytes);
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
    if (n < kMaxSpaces) {
      p.spaces.push_back(w);
      return;
    }
  }
  destroy(w);
}

}  // namespace qs
