// qs_small.hip -- gate runs on registers that fit one compute unit's LDS.
//
// A register of up to 2^13 complex128 amplitudes (128 KiB) is one sweep tile
// or a few: k_sweep runs it on one to four workgroups, one wave per SIMD, and
// every op is a chain of latencies there (the op's record and matrix fetched
// from memory, its code, hundreds of instructions of its own, fetched through
// the instruction cache): 2.1 us per op at 12 qubits against 0.21 us of FP64
// issue.  Below one tile it is a kernel launch per gate.  Here one workgroup
// of up to 16 waves loads the state into LDS once, runs the whole list of
// gates on it and stores it once.  The list comes in passes: two 2x2s (each
// with a matrix for the amplitudes where its pattern of control bits holds
// and one, or none, for the others) on quads of amplitudes, one 4x4, or up to
// eight phases; one small body of code serves them all, so it stays in the
// instruction cache, and the passes' records come through LDS in chunks of 32,
// each loaded before its passes run.  What bounds it is LDS: 0.65 us a pass on
// 4096 complex128 amplitudes, 0.43 us of it to read and write them.
// 12 qubits, 460 gates (complex128): 240 us, 484 us as two sweeps; a run of
// one-qubit gates on 3 qubits: 3.1 us, 4 kernels of 1.4 us and their gaps.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdlib>
#include <cstring>
#include <deque>
#include <type_traits>
#include <vector>

#include "qs_sweep.h"
#include "qs_sweep_kernel.h"
#include "qs_sweep_merge.h"

namespace qs {
namespace {

using namespace qs::merge;

constexpr int kSmallThreads = 1024;
constexpr int kSmallPhases = 8;
constexpr int kSmallMost = 13;  // qubits, complex128

enum : uint32_t { SM_PAIR = 1, SM_DENSE2 = 2, SM_PHASES = 3 };
// flags of the 2x2 in place j of a pair pass
enum : uint32_t {
  SF_ELSE = 1,       // has a matrix for where the pattern fails (else: untouched)
  SF_OWN_FIRST = 2,  // the second output adds its own amplitude's term first
};

// One pass.  SM_PAIR: 2x2 j on bit t[j], m[16 j ..) the matrix where (i & cm)
// == cv and m[16 j + 8 ..) the other one (row-major {re, im}); count 1 or 2.
// SM_DENSE2: the 4x4 m on bits t[0] (low matrix bit) and t[1] where (i &
// cm[0]) == cv[0].  SM_PHASES: `count` values m[2 j], m[2 j + 1] with pattern
// cm[j], cv[j].
template <typename R>
struct SmallPass {
  uint32_t kind, count, t[2];
  uint32_t flags[2], pad[2];
  uint32_t cm[kSmallPhases], cv[kSmallPhases];
  R m[32];
};

template <typename R>
constexpr int kChunkPasses = 32;  // 11 KiB (complex128), 7 KiB per chunk

// LDS position of amplitude j (as rev_pos of the reverse blocks): strided
// accesses of a pass on low bits spread over the banks; linear over XOR.
__device__ __forceinline__ uint32_t small_pos(uint32_t j) { return j ^ ((j >> 3) & 7u); }

__device__ __forceinline__ uint32_t small_insert0(uint32_t p, uint32_t q) {
  return p + (p & ~((1u << q) - 1u));
}

// acc + (mr + i mi) a, the multiply-adds in the order of the per-gate kernels.
template <typename R, typename T>
__device__ __forceinline__ T small_cmla(T acc, R mr, R mi, T a) {
  acc.x = fma(mr, a.x, acc.x);
  acc.x = fma(-mi, a.y, acc.x);
  acc.y = fma(mr, a.y, acc.y);
  acc.y = fma(mi, a.x, acc.y);
  return acc;
}

// The 2x2 in place j of a pass on the pair (x, y) at index i (bit t clear).
template <typename R, typename T>
__device__ __forceinline__ void small_2x2(const SmallPass<R> &p, int j, uint32_t flags, uint32_t cm,
                                          uint32_t cv, uint32_t i, T &x, T &y) {
  const bool on = (i & cm) == cv;
  if (!on && !(flags & SF_ELSE)) return;
  const R *m = p.m + 16 * j + (on ? 0 : 8);
  const T z = {0, 0};
  const T u = small_cmla(small_cmla(z, m[0], m[1], x), m[2], m[3], y);
  const T w = (flags & SF_OWN_FIRST)
                  ? small_cmla(small_cmla(z, m[6], m[7], y), m[4], m[5], x)
                  : small_cmla(small_cmla(z, m[4], m[5], x), m[6], m[7], y);
  x = u;
  y = w;
}

// A list short enough for the kernel's arguments (at most 4 KiB): no copy of
// its own to the device, 3 us of the stream and 4 of the host.
template <typename R>
constexpr int kArgPasses = sizeof(R) == 8 ? 8 : 14;

template <typename R, int N>
struct SmallArgs {
  SmallPass<R> p[N > 0 ? N : 1];
};

// One workgroup; 2^n amplitudes (n >= 2) in dynamic LDS, then the chunk.  The
// passes are in `args` (NA > 0) or at prog.
template <typename R, int NA>
__global__ __launch_bounds__(kSmallThreads) void k_small(typename sweep::SV2<R>::T *__restrict__ psi,
                                                         int n, const SmallPass<R> *__restrict__ prog,
                                                         int npass, uint32_t basis,
                                                         SmallArgs<R, NA> args) {
  using T = typename sweep::SV2<R>::T;
  extern __shared__ unsigned char small_smem[];
  T *s = (T *)small_smem;
  const uint32_t N = 1u << n;
  SmallPass<R> *chunk = (SmallPass<R> *)(small_smem + (size_t)N * sizeof(T));
  const uint32_t tid = threadIdx.x, nt = blockDim.x;
  // (basis < 2^n: the state is that basis state and not in memory yet)
  if (basis < N)
    for (uint32_t i = tid; i < N; i += nt) s[small_pos(i)] = T{(R)(i == basis), 0};
  else
    for (uint32_t i = tid; i < N; i += nt) s[small_pos(i)] = psi[i];
  constexpr int CP = kChunkPasses<R>;
  constexpr uint32_t kWords = CP * sizeof(SmallPass<R>) / 16;
  const uint4 *src = reinterpret_cast<const uint4 *>(NA > 0 ? args.p : prog);
  uint4 *dst = reinterpret_cast<uint4 *>(chunk);
  const uint32_t total = (uint32_t)npass * (uint32_t)(sizeof(SmallPass<R>) / 16);
  for (int c0 = 0; c0 < npass; c0 += CP) {
    // (every pass ends with a barrier: nobody reads the old chunk any more)
    const uint32_t w0 = (uint32_t)c0 * (uint32_t)(sizeof(SmallPass<R>) / 16);
    for (uint32_t w = tid; w < kWords && w0 + w < total; w += nt) dst[w] = src[w0 + w];
    __syncthreads();
    const int cn = npass - c0 < CP ? npass - c0 : CP;
    for (int c = 0; c < cn; ++c) {
      const SmallPass<R> &p = chunk[c];
      const uint32_t kind = __builtin_amdgcn_readfirstlane(p.kind);
      const uint32_t count = __builtin_amdgcn_readfirstlane(p.count);
      if (kind == SM_PHASES) {
        for (uint32_t i = tid; i < N; i += nt) {
          T a = s[small_pos(i)];
          bool any = false;
          for (uint32_t j = 0; j < count; ++j) {
            if ((i & p.cm[j]) != p.cv[j]) continue;
            a = small_cmla(T{0, 0}, p.m[2 * j], p.m[2 * j + 1], a);
            any = true;
          }
          if (any) s[small_pos(i)] = a;
        }
      } else {
        const uint32_t ta = __builtin_amdgcn_readfirstlane(p.t[0]);
        const uint32_t tb = __builtin_amdgcn_readfirstlane(p.t[1]);
        const uint32_t b1 = 1u << ta, b2 = 1u << tb;
        const uint32_t p1 = small_pos(b1), p2 = small_pos(b2);
        const uint32_t lo = ta < tb ? ta : tb, hi = ta < tb ? tb : ta;
        const uint32_t f0 = __builtin_amdgcn_readfirstlane(p.flags[0]);
        const uint32_t f1 = __builtin_amdgcn_readfirstlane(p.flags[1]);
        const uint32_t cm0 = __builtin_amdgcn_readfirstlane(p.cm[0]);
        const uint32_t cv0 = __builtin_amdgcn_readfirstlane(p.cv[0]);
        const uint32_t cm1 = __builtin_amdgcn_readfirstlane(p.cm[1]);
        const uint32_t cv1 = __builtin_amdgcn_readfirstlane(p.cv[1]);
        for (uint32_t q = tid; q < N / 4; q += nt) {
          const uint32_t i = small_insert0(small_insert0(q, lo), hi);
          const uint32_t a0 = small_pos(i), a1 = a0 ^ p1, a2 = a0 ^ p2, a3 = a1 ^ p2;
          T v0 = s[a0], v1 = s[a1], v2 = s[a2], v3 = s[a3];
          if (kind == SM_PAIR) {
            small_2x2(p, 0, f0, cm0, cv0, i, v0, v1);
            small_2x2(p, 0, f0, cm0, cv0, i | b2, v2, v3);
            if (count == 2) {
              small_2x2(p, 1, f1, cm1, cv1, i, v0, v2);
              small_2x2(p, 1, f1, cm1, cv1, i | b1, v1, v3);
            }
          } else if ((i & cm0) == cv0) {
            const T in[4] = {v0, v1, v2, v3};
            T out[4];
#pragma unroll
            for (int r = 0; r < 4; ++r) {
              out[r] = T{0, 0};
#pragma unroll
              for (int k = 0; k < 4; ++k)
                out[r] = small_cmla(out[r], p.m[8 * r + 2 * k], p.m[8 * r + 2 * k + 1], in[k]);
            }
            v0 = out[0];
            v1 = out[1];
            v2 = out[2];
            v3 = out[3];
          }
          s[a0] = v0;
          s[a1] = v1;
          s[a2] = v2;
          s[a3] = v3;
        }
      }
      __syncthreads();
    }
  }
  if (npass == 0) __syncthreads();
  for (uint32_t i = tid; i < N; i += nt) psi[i] = s[small_pos(i)];
}

// Whether QS_GATE1_LANE keeps the lane form of one-qubit gates (default on),
// whose order of additions complex64 follows here.
bool lane_form() {
  static const bool on = [] {
    const char *v = std::getenv("QS_GATE1_LANE");
    return !(v && v[0] == '0');
  }();
  return on;
}

template <typename R>
struct Builder {
  std::vector<SmallPass<R>> prog;
  int n;
  bool open = false;  // the last pass is a pair with room for a second 2x2

  static void put(R *m, const cd *v, int count) {
    for (int k = 0; k < count; ++k) {
      m[2 * k] = (R)v[k].re;
      m[2 * k + 1] = (R)v[k].im;
    }
  }

  SmallPass<R> &add(uint32_t kind) {
    prog.push_back(SmallPass<R>{});
    prog.back().kind = kind;
    open = false;
    return prog.back();
  }

  // m1 where (i & pm) == pv, m0 (null: untouched) elsewhere, on bit t.
  void two(int t, uint64_t pm, uint64_t pv, const cd *m1, const cd *m0, bool own_first) {
    int j = 0;
    if (open && (int)prog.back().t[0] != t) {
      j = 1;
      open = false;
    } else {
      add(SM_PAIR);
      open = true;
    }
    SmallPass<R> &p = prog.back();
    p.count = (uint32_t)(j + 1);
    p.t[j] = (uint32_t)t;
    if (j == 0) p.t[1] = t == 0 ? 1u : 0u;  // the quads' other bit
    p.flags[j] = (m0 ? SF_ELSE : 0u) | (own_first ? SF_OWN_FIRST : 0u);
    p.cm[j] = (uint32_t)pm;
    p.cv[j] = (uint32_t)pv;
    put(p.m + 16 * j, m1, 4);
    if (m0) put(p.m + 16 * j + 8, m0, 4);
  }

  void phase(uint64_t pm, uint64_t pv, const cd &v) {
    if (prog.empty() || prog.back().kind != SM_PHASES || prog.back().count == kSmallPhases)
      add(SM_PHASES);
    SmallPass<R> &p = prog.back();
    p.cm[p.count] = (uint32_t)pm;
    p.cv[p.count] = (uint32_t)pv;
    put(p.m + 2 * p.count, &v, 1);
    ++p.count;
  }

  static bool takes(const Gate &g) {
    if (g.bmask) return false;
    if (g.kind == Gate::kSparse) return true;
    return (g.kind == Gate::kDense || g.kind == Gate::kDiag) && g.na <= 2;
  }

  void gate(const Gate &g, bool exact) {
    if (g.kind == Gate::kSparse) {
      for (size_t e = 0; e < g.spat.size(); ++e) phase(g.smask, g.spat[e], g.m[e]);
    } else if (g.kind == Gate::kDiag) {
      for (size_t e = 0; e < g.m.size(); ++e) {
        uint64_t pm = g.cmask, pv = g.cval;
        for (int a = 0; a < g.na; ++a) {
          pm |= 1ull << g.act[a];
          if ((e >> a) & 1) pv |= 1ull << g.act[a];
        }
        phase(pm, pv, g.m[e]);
      }
    } else if (g.na == 1) {
      const bool own = exact && lane_form() && g.act[0] < 6 && n >= 6 && !(g.cmask & 0x3Full);
      two(g.act[0], g.cmask, g.cval, g.m.data(), nullptr, own);
    } else {
      SmallPass<R> &p = add(SM_DENSE2);
      p.count = 1;
      p.t[0] = (uint32_t)g.act[0];
      p.t[1] = (uint32_t)g.act[1];
      p.cm[0] = (uint32_t)g.cmask;
      p.cv[0] = (uint32_t)g.cval;
      put(p.m, g.m.data(), 16);
    }
  }
};

template <typename R>
hipError_t execute_small_t(SweepRunner &run, const std::vector<Gate> &gates, uint64_t *sweeps) {
  using T = typename sweep::SV2<R>::T;
  const int n = run.n;
  constexpr bool exact = std::is_same<R, float>::value;
  Builder<R> b;
  b.n = n;
  auto launch = [&]() -> hipError_t {
    if (b.prog.empty()) return hipSuccess;
    constexpr int NA = kArgPasses<R>;
    const bool in_args = b.prog.size() <= (size_t)NA;
    void *d = nullptr;
    hipError_t e = hipSuccess;
    if (!in_args) e = run.upload(b.prog.data(), b.prog.size() * sizeof(SmallPass<R>), &d);
    if (e != hipSuccess) return e;
    const size_t lds = (sizeof(T) << n) + kChunkPasses<R> * sizeof(SmallPass<R>);
    static const hipError_t set = [] {
      const hipError_t e1 = hipFuncSetAttribute(
          (const void *)k_small<R, 0>, hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
      const hipError_t e2 = hipFuncSetAttribute(
          (const void *)k_small<R, NA>, hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
      return e1 != hipSuccess ? e1 : e2;
    }();
    if (set != hipSuccess) return set;
    const unsigned threads = (unsigned)std::min(kSmallThreads, std::max(64, 1 << (n - 2)));
    if (run.mark) run.mark(true);
    const uint32_t basis = run.fresh ? (uint32_t)run.known_val : ~0u;
    if (in_args) {
      SmallArgs<R, NA> args{};
      std::memcpy(args.p, b.prog.data(), b.prog.size() * sizeof(SmallPass<R>));
      hipLaunchKernelGGL((k_small<R, NA>), dim3(1), dim3(threads), lds, run.stream, (T *)run.psi,
                         n, nullptr, (int)b.prog.size(), basis, args);
    } else {
      hipLaunchKernelGGL((k_small<R, 0>), dim3(1), dim3(threads), lds, run.stream, (T *)run.psi,
                         n, (const SmallPass<R> *)d, (int)b.prog.size(), basis,
                         SmallArgs<R, 0>{});
    }
    if (run.mark) run.mark(false);
    e = hipGetLastError();
    if (e == hipSuccess) {
      ++*sweeps;
      run.known = run.known_val = 0;
      run.fresh = false;
    }
    b.prog.clear();
    b.open = false;
    return e;
  };
  // merged like a sweep's ops (qs_sweep_merge.h); every qubit is on the tile
  // and no pattern is on a register slot.  Complex64 runs the gates as they
  // come, each rounded as its own kernel would round it.
  int slot[64];
  for (int q = 0; q < 64; ++q) slot[q] = q < n ? kFirstLaneSlot : -1;
  for (size_t at = 0; at < gates.size();) {
    // (one gate alone on the largest state: its own kernel's many workgroups
    // are faster than one's loads and stores: a 4x4 on 13 qubits 14.0 us with
    // its synchronisation, 18.2 here; on 12 qubits 15.6 here, 17.3)
    const bool alone = n >= kSmallMost && !run.fresh && gates.size() == 1;
    if (alone || !Builder<R>::takes(gates[at])) {
      hipError_t e = launch();
      if (e == hipSuccess) e = sweep_settle(run);
      if (e == hipSuccess) e = run.single(gates[at]);
      if (e != hipSuccess) return e;
      ++at;
      continue;
    }
    size_t end = at;
    while (end < gates.size() && Builder<R>::takes(gates[end])) ++end;
    std::vector<SweepOp> items(end - at);
    for (size_t k = at; k < end; ++k) items[k - at].g = &gates[k];
    if (!exact && sweep_merge_ops()) merge_sweep_ops<long double>(items, slot, 0);
    for (const SweepOp &o : items) {
      if (!o.alive) {
        if (run.merged) ++*run.merged;
        continue;
      }
      if (run.sweep_ops) ++*run.sweep_ops;
      if (o.g)
        b.gate(*o.g, exact);
      else
        b.two(o.t, o.pm, o.pv, o.m1, o.pm ? o.m0 : nullptr, false);
    }
    at = end;
    hipError_t e = launch();
    if (e != hipSuccess) return e;
  }
  return hipSuccess;
}

}  // namespace

// Complex128 up to 13 qubits (128 KiB of LDS; 12 qubits of 460 gates and 12
// measures take 855 us here and 1105 us as sweeps; 14 qubits would not fit,
// and fill four or more workgroups of a sweep).  Complex64 only where its
// gates would run as kernels of their own (registers smaller than a sweep
// tile: up to 10 qubits): its sweeps round in another order.
bool small_fits(int n, bool c64) {
  static const bool on = [] {
    const char *v = std::getenv("QS_SMALL");
    return !(v && v[0] == '0');
  }();
  if (!on || n < 2) return false;
  return c64 ? n < sweep::kLaneBits + sweep_reg_bits(true) : n <= kSmallMost;
}

hipError_t execute_small(SweepRunner &run, const std::vector<Gate> &gates, uint64_t *sweeps) {
  return run.dtype_c64 ? execute_small_t<float>(run, gates, sweeps)
                       : execute_small_t<double>(run, gates, sweeps);
}

}  // namespace qs
