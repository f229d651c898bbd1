// CPU check of the pool of kept device memory: qs_pool.hip itself, compiled
// against a stand-in for the HIP runtime (fake_hip).  The first argument
// names the check; prints "ok" or what failed.
#include <dlfcn.h>
#include <hip/hip_runtime.h>
#include <pthread.h>

#include <cerrno>
#include <chrono>
#include <cstdio>
#include <cstring>
#include <thread>

#include "qs_pool.hip"

using namespace qs;

// Thread creation, refused on demand.
static bool no_threads = false;
extern "C" int pthread_create(pthread_t *t, const pthread_attr_t *a, void *(*f)(void *), void *x) {
  if (no_threads) return EAGAIN;
  using Fn = int (*)(pthread_t *, const pthread_attr_t *, void *(*)(void *), void *);
  static const Fn next = reinterpret_cast<Fn>(dlsym(RTLD_NEXT, "pthread_create"));
  return next(t, a, f, x);
}

namespace {

constexpr size_t MiB = 1ull << 20, GiB = 1ull << 30;

#define CHECK(cond)                                                \
  do {                                                             \
    if (!(cond)) {                                                 \
      std::printf("line %d: %s\n", __LINE__, #cond);               \
      return 1;                                                    \
    }                                                              \
  } while (0)

void *take(size_t bytes, int device = 0) {
  void *p = nullptr;
  return pool_malloc(&p, bytes, device) == hipSuccess ? p : nullptr;
}

void wait_ms(int ms) { std::this_thread::sleep_for(std::chrono::milliseconds(ms)); }

// Until `cond`, at most `ms`.
template <typename F>
bool within(int ms, F &&cond) {
  for (; ms > 0 && !cond(); ms -= 10) wait_ms(10);
  return cond();
}

// A block goes to the next caller of its size; all kept ones together stay
// within an eighth of the device, the oldest leave first; a failed allocation
// gets what is kept.
int bounds() {
  void *a = take(GiB), *b = take(2 * GiB);
  CHECK(a && b);
  pool_free(a, GiB, 0);
  CHECK(fake::used(0) == 3 * GiB);
  CHECK(take(GiB) == a);
  void *c = take(GiB);
  CHECK(c && c != a);
  pool_free(a, GiB, 0);
  pool_free(b, 2 * GiB, 0);
  pool_free(c, GiB, 0);
  void *d = take(5 * GiB);
  pool_free(d, 5 * GiB, 0);  // 9 GiB would be kept: the oldest one leaves
  CHECK(fake::device_of(a) == -1 && fake::device_of(b) == 0 && fake::used(0) == 8 * GiB);
  void *e = take(9 * GiB);  // more than an eighth is not kept
  pool_free(e, 9 * GiB, 0);
  CHECK(fake::used(0) == 8 * GiB);
  void *f = take(60 * GiB);
  CHECK(f && fake::used(0) == 60 * GiB);
  CHECK(!take(60 * GiB));
  pool_free(f, 60 * GiB, 0);
  CHECK(fake::used(0) == 0);
  return 0;
}

// A block that nothing has taken for a second goes back, also while others
// come and go.
int idle() {
  void *big = take(4 * GiB);
  pool_free(big, 4 * GiB, 0);
  for (int k = 0; k < 200; ++k) {
    void *s = take(MiB);
    pool_free(s, MiB, 0);
    wait_ms(10);
  }
  CHECK(fake::device_of(big) == -1);
  CHECK(fake::used(0) == MiB);
  return 0;
}

// The idle thread frees while another thread records a stream: the recording
// (global mode) refuses every thread's allocations and frees that have not
// said otherwise.
int capture() {
  void *big = take(4 * GiB);
  fake::rt().capturing = true;
  pool_free(big, 4 * GiB, 0);
  CHECK(within(3000, [&] { return fake::device_of(big) == -1; }));
  CHECK(fake::rt().refused_frees == 0);
  CHECK(fake::mode == hipStreamCaptureModeGlobal);  // this thread's is as it was
  return 0;
}

// No thread to be had: nothing may throw out of pool_free (a C entry calls
// it), and what would never be given back is not kept.
int no_thread() {
  void *big = take(4 * GiB), *s = take(MiB);
  no_threads = true;
  pool_free(s, MiB, 0);
  pool_free(big, 4 * GiB, 0);
  CHECK(fake::used(0) <= 64 * MiB);
  no_threads = false;
  big = take(4 * GiB);
  pool_free(big, 4 * GiB, 0);  // the next one may start it
  CHECK(fake::device_of(big) == 0);
  CHECK(within(3000, [&] { return fake::device_of(big) == -1; }));
  return 0;
}

// An allocation that fails while another thread (first the one that hands a
// block in, then the idle one) is giving memory back waits for that.
int freeing() {
  void *a = take(5 * GiB), *b = take(6 * GiB), *rest = take(50 * GiB);
  pool_free(a, 5 * GiB, 0);
  fake::free_ms = 300;
  std::thread other([&] { pool_free(b, 6 * GiB, 0); });  // the 5 GiB leave
  wait_ms(100);
  fake::free_ms = 0;
  void *c = take(14 * GiB);  // needs both blocks' memory
  CHECK(c);
  other.join();
  CHECK(fake::device_of(a) == -1 && fake::device_of(b) == -1);
  pool_free(c, 14 * GiB, 0);
  a = take(5 * GiB);
  c = take(9 * GiB);
  CHECK(a && c);
  fake::free_ms = 600;
  pool_free(a, 5 * GiB, 0);
  wait_ms(1200);  // the idle thread frees it now
  CHECK(take(5 * GiB));
  CHECK(rest);
  return 0;
}

// Memory is its owner's device's, whatever device the calling thread has
// current (a register's buffers grow in calls made at any time).
int device() {
  fake::current = 1;
  void *a = take(GiB, 0);
  CHECK(fake::device_of(a) == 0 && fake::current == 1);
  pool_free(a, GiB, 0);
  void *b = take(GiB, 1);
  CHECK(fake::device_of(b) == 1 && b != a);
  fake::current = 0;
  pool_free(b, GiB, 1);
  CHECK(take(GiB, 0) == a && take(GiB, 1) == b);
  CHECK(!take(64 * GiB, 1) && fake::current == 0);
  return 0;
}

// Everything kept goes back when a program asks for it, also what the idle
// thread leaves and workspaces of closed registers; blocks in use stay.
int release() {
  Workspace *w[6];
  for (Workspace *&x : w) CHECK(workspace_get(&x, &x - w < 3 ? 0 : 1) == hipSuccess);
  void *a = take(MiB), *b = take(GiB), *mine = take(2 * GiB);
  pool_free(a, MiB, 0);
  pool_free(b, GiB, 0);
  for (Workspace *x : w) workspace_put(x);
  CHECK(fake::used(0) > 3 * GiB && fake::used(1) > 0);
  pool_release();
  CHECK(fake::used(0) == 2 * GiB && fake::used(1) == 0);
  CHECK(fake::device_of(mine) == 0 && fake::streams == 0 && fake::host_blocks == 0);
  CHECK(workspace_get(&w[0], 0) == hipSuccess);
  workspace_put(w[0]);
  return 0;
}

}  // namespace

int main(int argc, char **argv) {
  const char *what = argc > 1 ? argv[1] : "";
  int rc = 1;
  if (!std::strcmp(what, "bounds")) rc = bounds();
  if (!std::strcmp(what, "idle")) rc = idle();
  if (!std::strcmp(what, "capture")) rc = capture();
  if (!std::strcmp(what, "freeing")) rc = freeing();
  if (!std::strcmp(what, "device")) rc = device();
  if (!std::strcmp(what, "release")) rc = release();
  if (!std::strcmp(what, "no_thread")) rc = no_thread();
  if (rc == 0) std::printf("ok\n");
  return rc;
}
