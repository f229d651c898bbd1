// qs_kernels.hip -- per-gate kernels and FP64 reductions for gfx950.
//
// The per-gate kernels replace the hot loop of Register::try_apply_fast
// (src/register.rs:155-189): instead of filtering all 2^n indices and
// gathering each group through heap vectors, a thread expands a dense counter
// p over the free index bits into a group base index (inserting zeros at the
// sorted fixed bit positions: targets and controls), then reads, multiplies
// and writes the group in place.  Groups are disjoint, so in-place equals the
// reference's out-of-place copy.  Amplitudes whose control bits do not match
// are never touched, which is why a gate with c controls moves 2^(n-c)
// amplitudes instead of 2^n.
//
// Reductions (measure, norm, inner product, equality) accumulate in FP64 for
// both storage precisions, with a fixed grid so results are deterministic.
#include <algorithm>
#include <cstdlib>
#include <type_traits>
#include <utility>

#include "qs_internal.h"

namespace qs {

template <typename R>
struct V2;
template <>
struct V2<double> {
  using T = double2;
};
template <>
struct V2<float> {
  using T = float2;
};

Fixed make_fixed(uint64_t mask, uint64_t set) {
  Fixed f{};
  f.set = set;
  f.nf = 0;
  for (int b = 0; b < 64; ++b)
    if ((mask >> b) & 1ull) f.pos[f.nf++] = (uint8_t)b;
  return f;
}

__device__ __forceinline__ uint64_t expand(uint64_t p, const Fixed &f) {
  for (int i = 0; i < f.nf; ++i) {
    const uint64_t lo = p & ((1ull << f.pos[i]) - 1ull);
    p = ((p ^ lo) << 1) | lo;
  }
  return p | f.set;
}

template <typename T>
__device__ __forceinline__ T cmla(T acc, decltype(T::x) mr, decltype(T::x) mi, T a) {
  acc.x = fma(mr, a.x, acc.x);
  acc.x = fma(-mi, a.y, acc.x);
  acc.y = fma(mr, a.y, acc.y);
  acc.y = fma(mi, a.x, acc.y);
  return acc;
}

template <typename T>
__device__ __forceinline__ T czero() {
  T z;
  z.x = 0;
  z.y = 0;
  return z;
}

constexpr int kBlock = 256;

// Streaming access.  A state larger than the last-level cache (256 MiB
// Infinity Cache) is read and written once per gate, so the gate kernels
// load and store its amplitudes with the nontemporal hint.  Measured on a
// 16 GiB complex128 state, pair updates (i, i | 2^t) in place: 5.5-5.8 TB/s
// with the hint against 5.2-5.4 without for t >= 3, but 5.0 against 5.2 for
// t < 3, where a wave's two loads interleave inside the same 128-byte lines.
constexpr uint64_t kStreamBytes = 256ull << 20;

static bool streaming(int n, size_t amp_bytes) { return ((uint64_t)amp_bytes << n) > kStreamBytes; }

template <typename R>
struct NTV {
  typedef R T __attribute__((ext_vector_type(2)));
};

template <bool kNT, typename T>
__device__ __forceinline__ T ld(const T *p) {
  if constexpr (kNT) {
    using E = typename NTV<decltype(T::x)>::T;
    const E v = __builtin_nontemporal_load(reinterpret_cast<const E *>(p));
    T r;
    r.x = v.x;
    r.y = v.y;
    return r;
  } else {
    return *p;
  }
}

template <bool kNT, typename T>
__device__ __forceinline__ void st(T *p, T v) {
  if constexpr (kNT) {
    using E = typename NTV<decltype(T::x)>::T;
    E e;
    e.x = v.x;
    e.y = v.y;
    __builtin_nontemporal_store(e, reinterpret_cast<E *>(p));
  } else {
    *p = v;
  }
}

// Calls f(integral_constant<bool, nt>).
template <typename F>
static void nt_dispatch(bool nt, F &&f) {
  if (nt) f(std::integral_constant<bool, true>{});
  else f(std::integral_constant<bool, false>{});
}

// Read-only data every thread reads at the same address (gate matrices):
// through the constant address space the compiler keeps the reads scalar.
#define QS_KCONST __attribute__((address_space(4)))

static inline unsigned grid_for(uint64_t work, uint64_t per_block) {
  uint64_t g = (work + per_block - 1) / per_block;
  if (g < 1) g = 1;
  return (unsigned)g;
}

// ---- state initialisation ---------------------------------------------------

template <typename R>
__global__ __launch_bounds__(kBlock) void k_init_basis(typename V2<R>::T *psi, uint64_t len,
                                                       uint64_t k) {
  using T = typename V2<R>::T;
  for (uint64_t i = (uint64_t)blockIdx.x * kBlock + threadIdx.x; i < len;
       i += (uint64_t)gridDim.x * kBlock) {
    T v = czero<T>();
    if (i == k) v.x = 1;
    psi[i] = v;
  }
}

template <typename R>
__global__ __launch_bounds__(kBlock) void k_zero_outside(typename V2<R>::T *psi, uint64_t len,
                                                         uint64_t mask, uint64_t val) {
  using T = typename V2<R>::T;
  for (uint64_t i = (uint64_t)blockIdx.x * kBlock + threadIdx.x; i < len;
       i += (uint64_t)gridDim.x * kBlock)
    if ((i & mask) != val) psi[i] = czero<T>();
}

// Product state in the order of the kron fold of Register::new /
// try_from_qubits (src/register.rs:47-50, :94-96): amp = b_{n-1} * (... *
// (b_0 * 1)).
template <typename R>
__global__ __launch_bounds__(kBlock) void k_init_product(typename V2<R>::T *psi, int n,
                                                         ProductState p) {
  const double *q = p.q;
  using T = typename V2<R>::T;
  const uint64_t len = 1ull << n;
  for (uint64_t i = (uint64_t)blockIdx.x * kBlock + threadIdx.x; i < len;
       i += (uint64_t)gridDim.x * kBlock) {
    double ar = 1.0, ai = 0.0;
    for (int b = 0; b < n; ++b) {
      const int bit = (int)((i >> b) & 1ull);
      const double br = q[4 * b + 2 * bit], bi = q[4 * b + 2 * bit + 1];
      const double nr = br * ar - bi * ai;
      const double ni = br * ai + bi * ar;
      ar = nr;
      ai = ni;
    }
    T v;
    v.x = (R)ar;
    v.y = (R)ai;
    psi[i] = v;
  }
}

template <typename R>
hipError_t launch_init_basis(void *psi, int n, uint64_t k, hipStream_t s) {
  const uint64_t len = 1ull << n;
  unsigned g = grid_for(len, kBlock * 8);
  if (g > 65536) g = 65536;
  hipLaunchKernelGGL(k_init_basis<R>, dim3(g), dim3(kBlock), 0, s,
                     (typename V2<R>::T *)psi, len, k);
  return hipGetLastError();
}

template <typename R>
hipError_t launch_zero_outside(void *psi, int n, uint64_t mask, uint64_t val, hipStream_t s) {
  const uint64_t len = 1ull << n;
  unsigned g = grid_for(len, kBlock * 8);
  if (g > 65536) g = 65536;
  hipLaunchKernelGGL(k_zero_outside<R>, dim3(g), dim3(kBlock), 0, s, (typename V2<R>::T *)psi,
                     len, mask, val);
  return hipGetLastError();
}

template <typename R>
hipError_t launch_init_product(void *psi, int n, const ProductState &q, hipStream_t s) {
  const uint64_t len = 1ull << n;
  unsigned g = grid_for(len, kBlock * 8);
  if (g > 65536) g = 65536;
  hipLaunchKernelGGL(k_init_product<R>, dim3(g), dim3(kBlock), 0, s,
                     (typename V2<R>::T *)psi, n, q);
  return hipGetLastError();
}

// ---- dense gates --------------------------------------------------------------

template <typename R, int D>
struct MatArg {
  R re[D * D];
  R im[D * D];
};

// One active target (matrix bit 0 <-> qubit with stride `tbit`).  Each thread
// owns kItems units spaced one block apart, so a wave issues all its loads
// before the first multiply.  kX = 1: a unit is one pair (i, i | tbit).
// kX = 2: a unit is the two pairs at i and i | xbit, xbit a free index bit
// that fx also holds at 0, so a workgroup reads four streams (xbit 32 or 64
// KiB of amplitudes, as the host picks it; complex128 only).  Measured at 30 qubits,
// complex128, Haar gate, ms per launch: target 6-10 6.25-6.28 with kX = 1,
// 5.61-5.69 with kX = 2 and xbit = 2^12; target 13-29 6.00-6.10 against
// 5.37-5.53; target 11 5.27 against 5.22.  An xbit of 2^13 ran 6.0-6.9.
template <typename R, int kItems, bool kNT, int kX = 1>
__global__ __launch_bounds__(kBlock) void k_gate1(typename V2<R>::T *__restrict__ psi,
                                                  uint64_t npairs, Fixed fx, uint64_t tbit,
                                                  MatArg<R, 2> m, uint64_t xbit = 0) {
  using T = typename V2<R>::T;
  static_assert(kX == 1 || kX == 2, "kX: 1 or 2 pairs per unit");
  constexpr int NP = kItems * kX;
  const uint64_t base = (uint64_t)blockIdx.x * (kBlock * kItems) + threadIdx.x;
  T a0[NP], a1[NP];
  uint64_t i0[NP];
  bool ok[kItems];
#pragma unroll
  for (int it = 0; it < kItems; ++it) {
    const uint64_t p = base + (uint64_t)it * kBlock;
    ok[it] = p < npairs;
    if (ok[it]) {
      const uint64_t i = expand(p, fx);
#pragma unroll
      for (int x = 0; x < kX; ++x) {
        const int j = it * kX + x;
        i0[j] = x ? (i | xbit) : i;
        a0[j] = ld<kNT>(psi + i0[j]);
        a1[j] = ld<kNT>(psi + (i0[j] | tbit));
      }
    }
  }
#pragma unroll
  for (int j = 0; j < NP; ++j) {
    if (ok[j / kX]) {
      T r0 = czero<T>(), r1 = czero<T>();
      r0 = cmla(r0, m.re[0], m.im[0], a0[j]);
      r0 = cmla(r0, m.re[1], m.im[1], a1[j]);
      r1 = cmla(r1, m.re[2], m.im[2], a0[j]);
      r1 = cmla(r1, m.re[3], m.im[3], a1[j]);
      st<kNT>(psi + i0[j], r0);
      st<kNT>(psi + (i0[j] | tbit), r1);
    }
  }
}

// Partner lane l ^ 2^K of a 32-bit value by VALU cross-lane moves: DPP
// inside rows of 16 lanes for K < 4 -- quad_perm [1,0,3,2] (K = 0),
// [2,3,0,1] (K = 1), row_shl:4 into banks 0 and 2 plus row_shr:4 into banks
// 1 and 3 (K = 2: two independent moves, each writing the lanes the other
// leaves alone), row_ror:8 (K = 3) -- and gfx950's half swaps for K = 4, 5
// (a value swapped with itself: the first result holds the bit-clear half's
// values, the second the bit-set half's).
template <int K>
__device__ __forceinline__ int lane_partner(int v) {
  const bool hi = (threadIdx.x >> K) & 1;
  if constexpr (K == 0) return __builtin_amdgcn_mov_dpp(v, 0xB1, 0xF, 0xF, false);
  if constexpr (K == 1) return __builtin_amdgcn_mov_dpp(v, 0x4E, 0xF, 0xF, false);
  if constexpr (K == 2) {
    const int lo = __builtin_amdgcn_update_dpp(0, v, 0x104, 0xF, 0x5, false);  // row_shl:4
    return __builtin_amdgcn_update_dpp(lo, v, 0x114, 0xF, 0xA, false);        // row_shr:4
  }
  if constexpr (K == 3) return __builtin_amdgcn_mov_dpp(v, 0x128, 0xF, 0xF, false);
  if constexpr (K == 4) {
    const auto p = __builtin_amdgcn_permlane16_swap(v, v, false, false);
    return hi ? p[0] : p[1];
  }
  const auto p = __builtin_amdgcn_permlane32_swap(v, v, false, false);
  return hi ? p[0] : p[1];
}

template <int K>
__device__ __forceinline__ double lane_partner(double v) {
  const long long b = __double_as_longlong(v);
  const int lo = lane_partner<K>((int)(b & 0xffffffffll));
  const int hi = lane_partner<K>((int)(b >> 32));
  return __longlong_as_double(((long long)hi << 32) | (unsigned int)lo);
}

template <int K>
__device__ __forceinline__ float lane_partner(float v) {
  return __int_as_float(lane_partner<K>(__float_as_int(v)));
}

// One active target on qubit K < 6, controls (if any) on index bits >= 6:
// the pairs lie inside runs of 64 consecutive amplitudes, so k_gate1's two
// loads per pair would each touch every line at part occupancy.  Here lane
// l of a wave owns amplitude l of a run of 64 consecutive amplitudes (every
// load and store instruction is one contiguous 1 KiB / 512 B access), gets
// its partner's amplitude by DPP, and computes its own output with row
// ((l >> K) & 1) of the matrix.  Chunk c of 64 amplitudes is expand(c, fx)
// << 6 with fx holding the controls relative to bit 6.
//
// Chunk order (kStreams == 0): wave w takes chunks w * kItems + it.  With
// kStreams = S = 2^SB (nchunks a multiple of 2^(5 + SB)), a workgroup reads
// S streams 32 chunks apart: unit u = block * 4 * kItems + it * 4 + wave
// gives chunks (u mod 32) | (u / 32) << (5 + SB) | s << 5 for s < S.
// Measured at 30 qubits, complex128, gate on qubit 0: S = 4, kItems = 4
// (16 loads in flight per lane, 64 KiB per workgroup in four 16 KiB runs)
// 5.28 ms; one stream of 4 chunks per wave 5.92 ms; S = 2 5.55-5.70 ms;
// S = 8 5.42-5.96 ms; streams 16, 64 or 128 chunks apart 5.38-5.93 ms.
template <typename R, int K, int kItems, bool kNT, int kStreams = 0>
__global__ __launch_bounds__(kBlock) void k_gate1_lane(typename V2<R>::T *__restrict__ psi,
                                                       uint64_t nchunks, Fixed fx,
                                                       MatArg<R, 2> m) {
  using T = typename V2<R>::T;
  constexpr int S = kStreams > 0 ? kStreams : 1;
  constexpr int SB = S == 1 ? 0 : (S == 2 ? 1 : (S == 4 ? 2 : 3));
  static_assert(S == (1 << SB), "kStreams: 0, 1, 2, 4 or 8");
  constexpr int NL = kItems * S;
  const int lane = threadIdx.x & 63;
  const uint64_t wave = ((uint64_t)blockIdx.x * kBlock + threadIdx.x) >> 6;
  const bool hi = (lane >> K) & 1;
  // this lane's row: coefficient of its own amplitude (s) and the partner's (p)
  const R sr = hi ? m.re[3] : m.re[0], si = hi ? m.im[3] : m.im[0];
  const R pr = hi ? m.re[2] : m.re[1], pi = hi ? m.im[2] : m.im[1];
  T a[NL];
  uint64_t idx[NL];
  bool ok[NL];
#pragma unroll
  for (int it = 0; it < kItems; ++it) {
    if constexpr (kStreams == 0) {
      const uint64_t c = wave * kItems + it;
      ok[it] = c < nchunks;  // uniform over the wave: whole chunks only
      if (ok[it]) idx[it] = (expand(c, fx) << 6) | (uint64_t)lane;
    } else {
      // the workgroup's 4 * kItems * S chunks lie below nchunks as a whole or
      // not at all (the host launches nchunks / (4 * kItems * S) workgroups)
      const bool in = ((uint64_t)blockIdx.x + 1) * (4 * kItems * S) <= nchunks;
      const uint64_t u = (uint64_t)blockIdx.x * (4 * kItems) + it * 4 + (threadIdx.x >> 6);
      const uint64_t c0 = (u & 31ull) | ((u >> 5) << (5 + SB));
#pragma unroll
      for (int s = 0; s < S; ++s) {
        ok[it * S + s] = in;
        if (in) idx[it * S + s] = (expand(c0 | ((uint64_t)s << 5), fx) << 6) | (uint64_t)lane;
      }
    }
  }
#pragma unroll
  for (int j = 0; j < NL; ++j)
    if (ok[j]) a[j] = ld<kNT>(psi + idx[j]);
#pragma unroll
  for (int j = 0; j < NL; ++j) {
    if (ok[j]) {
      T y;
      y.x = lane_partner<K>(a[j].x);
      y.y = lane_partner<K>(a[j].y);
      T r = czero<T>();
      r = cmla(r, sr, si, a[j]);
      r = cmla(r, pr, pi, y);
      st<kNT>(psi + idx[j], r);
    }
  }
}

// Two active targets: quadruples (b, b|t0, b|t1, b|t0|t1) and a 4x4 matrix.
template <typename R, int kItems, bool kNT>
__global__ __launch_bounds__(kBlock) void k_gate2(typename V2<R>::T *__restrict__ psi,
                                                  uint64_t nquads, Fixed fx, uint64_t t0,
                                                  uint64_t t1, MatArg<R, 4> m) {
  using T = typename V2<R>::T;
  const uint64_t base = (uint64_t)blockIdx.x * (kBlock * kItems) + threadIdx.x;
#pragma unroll
  for (int it = 0; it < kItems; ++it) {
    const uint64_t p = base + (uint64_t)it * kBlock;
    if (p >= nquads) break;
    const uint64_t b = expand(p, fx);
    const uint64_t idx[4] = {b, b | t0, b | t1, b | t0 | t1};
    T a[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) a[j] = ld<kNT>(psi + idx[j]);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      T r = czero<T>();
#pragma unroll
      for (int j = 0; j < 4; ++j) r = cmla(r, m.re[4 * i + j], m.im[4 * i + j], a[j]);
      st<kNT>(psi + idx[i], r);
    }
  }
}

// Offset of row i of a group: the K bits of i deposited at the active
// positions (ax.pos[j] <- bit j of i).  Wave-uniform for uniform i.
template <int K>
__device__ __forceinline__ uint64_t row_offset(int i, const Fixed &ax) {
  uint64_t off = 0;
#pragma unroll
  for (int j = 0; j < K; ++j)
    if ((i >> j) & 1) off |= 1ull << ax.pos[j];
  return off;
}

// K = 3..5 active targets: one thread per group of D = 2^K amplitudes.  The
// thread loads its D amplitudes into registers, then computes and stores one
// output row at a time, out_i = sum_j M[i][j] a_j, so the D inputs are never
// overwritten before all rows are done (in place is safe: groups are
// disjoint).  The matrix (row-major {re, im}, the same for every thread) is
// read through the constant address space: its entries arrive on scalar
// loads and enter the FMAs as scalar operands, so the only per-amplitude
// memory traffic is the state itself.  Consecutive threads take consecutive
// groups, i.e. consecutive free index bits: with the low qubits free, each
// of the D loads of a wave is a run of 64 consecutive amplitudes.
// kReal: every matrix entry is real (Hadamard transforms, permutations,
// RY products), so a complex MAC is 2 FMAs instead of 4.
template <typename R, int K, bool kReal, bool kNT>
__global__ __launch_bounds__(kBlock) void k_gatek(typename V2<R>::T *__restrict__ psi,
                                                  uint64_t ngroups, Fixed fx, Fixed ax,
                                                  const R *__restrict__ m_g) {
  using T = typename V2<R>::T;
  constexpr int D = 1 << K;
  const QS_KCONST R *m = (const QS_KCONST R *)m_g;
  const uint64_t g = (uint64_t)blockIdx.x * kBlock + threadIdx.x;
  if (g >= ngroups) return;
  const uint64_t base = expand(g, fx);
  R ar[D], ai[D];
#pragma unroll
  for (int j = 0; j < D; ++j) {
    const T v = ld<kNT>(psi + (base | row_offset<K>(j, ax)));
    ar[j] = v.x;
    ai[j] = v.y;
  }
  for (int i = 0; i < D; ++i) {
    const QS_KCONST R *row = m + 2 * D * i;
    // two partial sums per component: independent FMA chains
    R sr0 = 0, si0 = 0, sr1 = 0, si1 = 0;
#pragma unroll
    for (int j = 0; j < D; j += 2) {
      const R mr0 = row[2 * j], mr1 = row[2 * j + 2];
      sr0 = fma(mr0, ar[j], sr0);
      si0 = fma(mr0, ai[j], si0);
      sr1 = fma(mr1, ar[j + 1], sr1);
      si1 = fma(mr1, ai[j + 1], si1);
      if constexpr (!kReal) {
        const R mi0 = row[2 * j + 1], mi1 = row[2 * j + 3];
        sr0 = fma(-mi0, ai[j], sr0);
        si0 = fma(mi0, ar[j], si0);
        sr1 = fma(-mi1, ai[j + 1], sr1);
        si1 = fma(mi1, ar[j + 1], si1);
      }
    }
    T out;
    out.x = sr0 + sr1;
    out.y = si0 + si1;
    st<kNT>(psi + (base | row_offset<K>(i, ax)), out);
  }
}

// Complex64 5-qubit blocks on the matrix cores.  Per wave, 64 groups (32
// amplitudes each) as the real product OUT = W x IN, with W the 64 x 64 real
// form [[Mr, -Mi], [Mi, Mr]] of the 32 x 32 complex matrix and IN the 64 x 64
// matrix of the groups' {re, im} components, by v_mfma_f32_32x32x2f32: two
// column blocks of 32 groups x two output row blocks (re, im) x 32 steps of
// K = 2 = 128 instructions per 2048 amplitudes.  FP32 matrix issue is twice
// the non-packed FP32 vector rate (157.3 against 78.6 TFLOP/s on MI355X),
// which the complex VALU form of k_gatek<float, 5> needs to reach the memory
// time.
//
// Operand layouts of the instruction (one 32 x 32 block): lane l holds
// A[l % 32][l / 32] and B[l / 32][l % 32]; accumulator register v of lane l
// holds D[(v % 4) + 8 (v / 4) + 4 (l / 32)][l % 32].  Lane l loads row m of
// group l, so every load instruction reads 64 consecutive groups (the 6
// lowest index bits are free).  A half swap (v_permlane32_swap) of rows 2t
// and 2t + 1 then leaves rows 2t (lanes 0..31) and 2t + 1 (lanes 32..63) of
// groups 0..31 in the first register, of groups 32..63 in the second: the B
// operands of step t (real parts; step 16 + t: imaginary parts) of the two
// column blocks.  The same swap of the two column blocks' accumulators gives
// rows i and i + 4 of all 64 groups, stored 64 consecutive groups at a time.
// W's A operands (64 per lane, one per instruction) are read once per
// persistent wave from the row-major matrix.
typedef float qs_floatx16 __attribute__((ext_vector_type(16)));

__device__ __forceinline__ void half32_swap(float &x, float &y) {
  const auto p = __builtin_amdgcn_permlane32_swap(__float_as_int(x), __float_as_int(y), false,
                                                  false);
  x = __int_as_float(p[0]);
  y = __int_as_float(p[1]);
}

template <bool kNT>
__global__ __launch_bounds__(64) void k_gatek5_mfma(float2 *__restrict__ psi, uint64_t nchunks,
                                                    Fixed fx, Fixed ax,
                                                    const float *__restrict__ m) {
  const int lane = threadIdx.x;
  const int h = lane >> 5, j = lane & 31;
  float aop0[32], aop1[32];  // W rows 0..31 (re out) and 32..63 (im out)
#pragma unroll
  for (int t = 0; t < 32; ++t) {
    const int c = 2 * t + h;  // W column
    const int cc = c & 31;
    const float mr = m[2 * (32 * j + cc)], mi = m[2 * (32 * j + cc) + 1];
    aop0[t] = c < 32 ? mr : -mi;
    aop1[t] = c < 32 ? mi : mr;
  }
  for (uint64_t ch = blockIdx.x; ch < nchunks; ch += gridDim.x) {
    const uint64_t base = expand(ch * 64 + (uint64_t)lane, fx);
    // b[0][t], b[1][t]: B operands of step t for column blocks 0 and 1
    float b0[32], b1[32];
#pragma unroll
    for (int t = 0; t < 16; ++t) {
      const float2 x = ld<kNT>(psi + (base | row_offset<5>(2 * t, ax)));
      const float2 y = ld<kNT>(psi + (base | row_offset<5>(2 * t + 1, ax)));
      b0[t] = x.x;
      b1[t] = y.x;
      b0[16 + t] = x.y;
      b1[16 + t] = y.y;
      half32_swap(b0[t], b1[t]);
      half32_swap(b0[16 + t], b1[16 + t]);
    }
    qs_floatx16 d00 = {}, d01 = {}, d10 = {}, d11 = {};  // d[column block][re/im]
#pragma unroll
    for (int t = 0; t < 32; ++t) {
      d00 = __builtin_amdgcn_mfma_f32_32x32x2f32(aop0[t], b0[t], d00, 0, 0, 0);
      d01 = __builtin_amdgcn_mfma_f32_32x32x2f32(aop1[t], b0[t], d01, 0, 0, 0);
      d10 = __builtin_amdgcn_mfma_f32_32x32x2f32(aop0[t], b1[t], d10, 0, 0, 0);
      d11 = __builtin_amdgcn_mfma_f32_32x32x2f32(aop1[t], b1[t], d11, 0, 0, 0);
    }
#pragma unroll
    for (int v = 0; v < 16; ++v) {
      // rows i0 = (v % 4) + 8 (v / 4) and i0 + 4 of all 64 groups
      float r0 = d00[v], r1 = d10[v], i0 = d01[v], i1 = d11[v];
      half32_swap(r0, r1);
      half32_swap(i0, i1);
      const int row = (v & 3) + 8 * (v >> 2);
      float2 o;
      o.x = r0;
      o.y = i0;
      st<kNT>(psi + (base | row_offset<5>(row, ax)), o);
      o.x = r1;
      o.y = i1;
      st<kNT>(psi + (base | row_offset<5>(row + 4, ax)), o);
    }
  }
}

// The same with 32 groups per wave, for blocks whose lowest active bit is
// index bit 5 (so 64 consecutive groups would not be consecutive
// amplitudes): lane l = 32h + j serves group j and loads its rows 2t + h,
// which are directly the B operands of steps t (real parts) and 16 + t
// (imaginary parts); rows 2t and 2t + 1 then differ in bit 5, so each load
// instruction still reads 512 consecutive bytes.  Its outputs are rows
// (v % 4) + 8 (v / 4) + 4h of D0 (real) and D1 (imaginary).
template <bool kNT>
__global__ __launch_bounds__(64) void k_gatek5_mfma32(float2 *__restrict__ psi,
                                                      uint64_t nchunks, Fixed fx, Fixed ax,
                                                      const float *__restrict__ m) {
  const int lane = threadIdx.x;
  const int h = lane >> 5, j = lane & 31;
  float aop0[32], aop1[32];
#pragma unroll
  for (int t = 0; t < 32; ++t) {
    const int c = 2 * t + h;
    const int cc = c & 31;
    const float mr = m[2 * (32 * j + cc)], mi = m[2 * (32 * j + cc) + 1];
    aop0[t] = c < 32 ? mr : -mi;
    aop1[t] = c < 32 ? mi : mr;
  }
  for (uint64_t ch = blockIdx.x; ch < nchunks; ch += gridDim.x) {
    const uint64_t base = expand(ch * 32 + (uint64_t)j, fx);
    float br[16], bi[16];
#pragma unroll
    for (int t = 0; t < 16; ++t) {
      const float2 v = ld<kNT>(psi + (base | row_offset<5>(2 * t + h, ax)));
      br[t] = v.x;
      bi[t] = v.y;
    }
    qs_floatx16 d0 = {}, d1 = {};
#pragma unroll
    for (int t = 0; t < 32; ++t) {
      const float b = t < 16 ? br[t] : bi[t - 16];
      d0 = __builtin_amdgcn_mfma_f32_32x32x2f32(aop0[t], b, d0, 0, 0, 0);
      d1 = __builtin_amdgcn_mfma_f32_32x32x2f32(aop1[t], b, d1, 0, 0, 0);
    }
#pragma unroll
    for (int v = 0; v < 16; ++v) {
      float2 o;
      o.x = d0[v];
      o.y = d1[v];
      st<kNT>(psi + (base | row_offset<5>((v & 3) + 8 * (v >> 2) + 4 * h, ax)), o);
    }
  }
}

// Whether complex64 5-qubit blocks use k_gatek5_mfma (QS_GATEK_MFMA, default
// on); the VALU form k_gatek<float, 5, false> otherwise.
static bool gatek_mfma() {
  static const bool on = [] {
    const char *v = std::getenv("QS_GATEK_MFMA");
    return !(v && v[0] == '0');
  }();
  return on;
}

// Bit layout of one staged block of k_gatek_staged: 64 groups x 2^K rows =
// 2^(6+K) slots.  Slot bit b sits at state index bit pa[b] (the active
// positions and the block's 6 lowest free positions, ascending), so the
// lanes of a staging load vary the lowest index bits the block has.  gslot[k]
// is the slot bit that carries bit k of the group number, jslot[k] the slot
// bit that carries matrix bit k.
struct StageMap {
  uint8_t pa[16];
  uint8_t gslot[6];
  uint8_t jslot[8];
};

// LDS position of slot s: the low 5 bits are XORed with the next 5, which
// spreads both the staging pattern (lanes = consecutive slots) and the
// compute pattern (lanes = groups) over the banks.
__device__ __forceinline__ int stage_phys(int s) { return s ^ ((s >> 5) & 31); }

// K = 3..5 active targets (complex128: those that k_dense_tile does not take)
// when low index bits are fixed (active or controls): the direct kernel's
// loads would then stride by 2^(lowest free bit) amplitudes per lane.  One
// wave stages 64 groups through LDS with loads over the block's lowest index
// bits, each lane computes its own group from registers (matrix on scalar loads, as in k_gatek), writes its outputs
// back to its own slots, and the wave stores the block the way it loaded it.
template <typename R, int K, bool kReal, bool kNT>
__global__ __launch_bounds__(64) void k_gatek_staged(typename V2<R>::T *__restrict__ psi,
                                                     uint64_t ngroups, Fixed fx, StageMap sm,
                                                     const R *__restrict__ m_g) {
  using T = typename V2<R>::T;
  constexpr int D = 1 << K;
  constexpr int kSlots = 64 * D;
  __shared__ T sl[kSlots];
  const QS_KCONST R *m = (const QS_KCONST R *)m_g;
  const int lane = threadIdx.x;
  const uint64_t g0 = (uint64_t)blockIdx.x * 64;
  if (g0 >= ngroups) return;  // whole blocks only: ngroups is a multiple of 64
  const uint64_t block_base = expand(g0, fx);
  // address bits of this lane's low 6 slot bits
  uint64_t lp = 0;
#pragma unroll
  for (int b = 0; b < 6; ++b)
    if ((lane >> b) & 1) lp |= 1ull << sm.pa[b];
#pragma unroll
  for (int r = 0; r < D; ++r) {
    uint64_t rp = 0;  // uniform: address bits of slot bits 6.. (value r)
#pragma unroll
    for (int b = 0; b < K; ++b)
      if ((r >> b) & 1) rp |= 1ull << sm.pa[6 + b];
    sl[stage_phys(r * 64 + lane)] = ld<kNT>(psi + (block_base | lp | rp));
  }
  __syncthreads();
  int tp = 0;  // this lane's group number on the slot bits
#pragma unroll
  for (int k = 0; k < 6; ++k)
    if ((lane >> k) & 1) tp |= 1 << sm.gslot[k];
  R ar[D], ai[D];
#pragma unroll
  for (int j = 0; j < D; ++j) {
    int jp = 0;
#pragma unroll
    for (int k = 0; k < K; ++k)
      if ((j >> k) & 1) jp |= 1 << sm.jslot[k];
    const T v = sl[stage_phys(tp | jp)];
    ar[j] = v.x;
    ai[j] = v.y;
  }
  for (int i = 0; i < D; ++i) {
    const QS_KCONST R *row = m + 2 * D * i;
    R sr0 = 0, si0 = 0, sr1 = 0, si1 = 0;
#pragma unroll
    for (int j = 0; j < D; j += 2) {
      const R mr0 = row[2 * j], mr1 = row[2 * j + 2];
      sr0 = fma(mr0, ar[j], sr0);
      si0 = fma(mr0, ai[j], si0);
      sr1 = fma(mr1, ar[j + 1], sr1);
      si1 = fma(mr1, ai[j + 1], si1);
      if constexpr (!kReal) {
        const R mi0 = row[2 * j + 1], mi1 = row[2 * j + 3];
        sr0 = fma(-mi0, ai[j], sr0);
        si0 = fma(mi0, ar[j], si0);
        sr1 = fma(-mi1, ai[j + 1], sr1);
        si1 = fma(mi1, ar[j + 1], si1);
      }
    }
    int ip = 0;
#pragma unroll
    for (int k = 0; k < K; ++k)
      if ((i >> k) & 1) ip |= 1 << sm.jslot[k];
    T out;
    out.x = sr0 + sr1;
    out.y = si0 + si1;
    sl[stage_phys(tp | ip)] = out;  // own slot: already read into registers
  }
  __syncthreads();
#pragma unroll
  for (int r = 0; r < D; ++r) {
    uint64_t rp = 0;
#pragma unroll
    for (int b = 0; b < K; ++b)
      if ((r >> b) & 1) rp |= 1ull << sm.pa[6 + b];
    st<kNT>(psi + (block_base | lp | rp), sl[stage_phys(r * 64 + lane)]);
  }
}

static uint64_t fx_mask(const Fixed &fx) {
  uint64_t m = 0;
  for (int i = 0; i < fx.nf; ++i) m |= 1ull << fx.pos[i];
  return m;
}

// The staged layout for a gate: active positions `ax` (matrix-bit order) and
// the lowest 6 free positions of `fx`.  Returns false when fewer than 6 free
// positions exist (tiny registers use the direct kernel).
static bool stage_map(const Fixed &fx, const Fixed &ax, int n, StageMap &sm) {
  uint64_t fixed = 0;
  for (int i = 0; i < fx.nf; ++i) fixed |= 1ull << fx.pos[i];
  uint64_t act = 0;
  for (int j = 0; j < ax.nf; ++j) act |= 1ull << ax.pos[j];
  uint64_t free6 = 0;
  int nfree = 0;
  for (int q = 0; q < n && nfree < 6; ++q)
    if (!((fixed >> q) & 1ull)) {
      free6 |= 1ull << q;
      ++nfree;
    }
  if (nfree < 6) return false;
  const uint64_t P = act | free6;
  int b = 0, gk = 0;
  uint8_t slot_of[64];
  for (int q = 0; q < 64; ++q)
    if ((P >> q) & 1ull) {
      slot_of[q] = (uint8_t)b;
      sm.pa[b++] = (uint8_t)q;
      if ((free6 >> q) & 1ull) sm.gslot[gk++] = (uint8_t)(b - 1);
    }
  // pa[] must list the slot bits low to high: slots 0..5 are the lowest six
  // positions of P and feed the lanes; the rest follow in order.
  for (int j = 0; j < ax.nf; ++j) sm.jslot[j] = slot_of[ax.pos[j]];
  return true;
}

template <typename R, int D>
static MatArg<R, D> to_matarg(const Gate &g) {
  MatArg<R, D> m;
  for (int e = 0; e < D * D; ++e) {
    m.re[e] = (R)g.m[e].re;
    m.im[e] = (R)g.m[e].im;
  }
  return m;
}

// Active positions in matrix-bit order (not sorted): pos[j] = act[j].
static Fixed active_positions(const Gate &g) {
  Fixed a{};
  a.nf = g.na;
  a.set = 0;
  for (int j = 0; j < g.na; ++j) a.pos[j] = (uint8_t)g.act[j];
  return a;
}

static uint64_t active_mask(const Gate &g) {
  uint64_t m = 0;
  for (int j = 0; j < g.na; ++j) m |= 1ull << g.act[j];
  return m;
}

// ---- dense blocks on the FP64 matrix cores -----------------------------------

typedef double f64x4 __attribute__((ext_vector_type(4)));

// Complex sums of 16 rows x 16 columns.  Four real sums, so that each is one
// chain over the summed index, as short as the halves of k_gatek's.
struct CplxAcc {
  f64x4 rr, ii, ri, ir;
  __device__ __forceinline__ void clear() { rr = ii = ri = ir = f64x4{0, 0, 0, 0}; }
  __device__ __forceinline__ double2 at(int v) const {
    return double2{rr[v] - ii[v], ri[v] + ir[v]};
  }
};

// acc += A x B for 4 values of the summed index: lane l holds A[l % 16][l / 16]
// and B[l / 16][l % 16]; element v of a sum, lane l, is [4 v + l / 16][l % 16].
template <bool kReal>
__device__ __forceinline__ void mfma_cplx(CplxAcc &s, double ar, double ai, double2 b) {
  s.rr = __builtin_amdgcn_mfma_f64_16x16x4f64(ar, b.x, s.rr, 0, 0, 0);
  s.ri = __builtin_amdgcn_mfma_f64_16x16x4f64(ar, b.y, s.ri, 0, 0, 0);
  if constexpr (!kReal) {
    s.ii = __builtin_amdgcn_mfma_f64_16x16x4f64(ai, b.y, s.ii, 0, 0, 0);
    s.ir = __builtin_amdgcn_mfma_f64_16x16x4f64(ai, b.x, s.ir, 0, 0, 0);
  }
}

// Bit layout of one tile of k_dense_tile: 2^LC groups (columns) x 2^K rows =
// 2^(K+LC) slots.  Slot bit b sits at state index bit pa[b], ascending (the
// active positions and the lowest LC free ones, so that consecutive lanes of
// a staging load take the lowest index bits the tile has); col[] and row[]
// are the slot bits of the column and of the row number.
struct TileMap {
  uint8_t pa[16];
  uint8_t col[8];
  uint8_t row[8];
};

// LDS place of slot s: the low four bits (16 complex128 cover the banks once)
// XORed with the next eight, so that 16 columns spread over the banks on
// whatever slot bits they are.  Linear over XOR.
__device__ __forceinline__ int tile_phys(int s) { return s ^ (((s >> 4) ^ (s >> 8)) & 15); }

// K = 4..6 active targets, complex128, in place.  A workgroup stages a tile
// through LDS and multiplies it by the 2^K x 2^K matrix: each of the 4 waves
// holds 16 rows of it in registers for all its tiles and computes NCT blocks
// of 16 columns.  The next tile's loads are in flight meanwhile.  Small tiles
// (16 or 32 KiB) keep several workgroups per CU and fill the chip from 15
// qubits on.  Bound by memory for K = 4 and 5, by the matrix cores' FP64 rate
// for K = 6: 27 qubits, 6 targets 1.2 ms a gate (57 TFLOP/s, 3.6 TB/s), 29.6
// ms with one thread per output; 5 targets with low qubits among them 0.80 ms
// (all low) to 1.02 ms (the others spread over far bits), 1.17 ms in
// k_gatek_staged; 15 qubits, 5 targets 4.9 us, 36 us in k_gatek.
template <int K, int LC, bool kReal, bool kNT>
__global__ __launch_bounds__(256, 2) void k_dense_tile(double2 *__restrict__ psi, uint64_t ntiles,
                                                       Fixed fx, TileMap tm,
                                                       const double2 *__restrict__ m) {
  constexpr int D = 1 << K, S = 1 << (K + LC);
  constexpr int RB = D / 16, CB = (1 << LC) / 16, NCT = RB * CB / 4;
  constexpr int KS = D / 4, NL = S / 256;
  static_assert(RB <= 4 && NCT >= 1, "four waves share the tile's blocks");
  __shared__ double2 lds[S];
  const int tid = threadIdx.x, lane = tid & 63, c = lane & 15, q = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r0 = 16 * (wave % RB), ct0 = (wave / RB) * NCT;
  // this thread's slots are tid + 256 r
  uint64_t lp = 0;
#pragma unroll
  for (int b = 0; b < 8; ++b)
    if ((tid >> b) & 1) lp |= 1ull << tm.pa[b];
  auto rp = [&](int r) {
    uint64_t v = 0;
#pragma unroll
    for (int b = 0; b < K + LC - 8; ++b)
      if ((r >> b) & 1) v |= 1ull << tm.pa[8 + b];
    return v;
  };
  int lcol = 0;  // this lane's column and low row bits, as LDS places
#pragma unroll
  for (int b = 0; b < 4; ++b)
    if ((c >> b) & 1) lcol |= 1 << tm.col[b];
  int lrow = 0;
#pragma unroll
  for (int b = 0; b < 2; ++b)
    if ((q >> b) & 1) lrow |= 1 << tm.row[b];
  const int at = tile_phys(lcol | lrow);
  auto row_at = [&](int s) {  // row bits from 2 up
    int v = 0;
#pragma unroll
    for (int b = 0; b < K - 2; ++b)
      if ((s >> b) & 1) v ^= tile_phys(1 << tm.row[2 + b]);
    return v;
  };
  auto col_at = [&](int s) {  // column bits from 4 up
    int v = 0;
#pragma unroll
    for (int b = 0; b < LC - 4; ++b)
      if ((s >> b) & 1) v ^= tile_phys(1 << tm.col[4 + b]);
    return v;
  };
  double ar[KS], ai[KS];
#pragma unroll
  for (int s = 0; s < KS; ++s) {
    const double2 v = m[(r0 + c) * D + 4 * s + q];
    ar[s] = v.x;
    ai[s] = v.y;
  }
  double2 next[NL];
  uint64_t t = blockIdx.x, base = 0;
  if (t < ntiles) {
    base = expand(t << LC, fx) | lp;
#pragma unroll
    for (int r = 0; r < NL; ++r) next[r] = ld<kNT>(psi + (base | rp(r)));
  }
  while (t < ntiles) {
#pragma unroll
    for (int r = 0; r < NL; ++r) lds[tile_phys(r * 256 + tid)] = next[r];
    __syncthreads();
    const uint64_t here = base;
    t += gridDim.x;
    if (t < ntiles) {
      base = expand(t << LC, fx) | lp;
#pragma unroll
      for (int r = 0; r < NL; ++r) next[r] = ld<kNT>(psi + (base | rp(r)));
    }
    CplxAcc acc[NCT];
#pragma unroll
    for (int j = 0; j < NCT; ++j) acc[j].clear();
#pragma unroll
    for (int s = 0; s < KS; ++s) {
      const int as = at ^ row_at(s);
#pragma unroll
      for (int j = 0; j < NCT; ++j) {
        const double2 b = lds[as ^ col_at(ct0 + j)];
        mfma_cplx<kReal>(acc[j], ar[s], ai[s], b);
      }
    }
    __syncthreads();  // every wave has read the inputs
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const int as = at ^ row_at(r0 / 4 + v);
#pragma unroll
      for (int j = 0; j < NCT; ++j) lds[as ^ col_at(ct0 + j)] = acc[j].at(v);
    }
    __syncthreads();
    // (the next tile goes to the places that this thread reads here)
#pragma unroll
    for (int r = 0; r < NL; ++r) st<kNT>(psi + (here | rp(r)), lds[tile_phys(r * 256 + tid)]);
  }
}

// Index bits of row or column number k of a matrix on the positions of ax.
__device__ __forceinline__ uint64_t deposit(uint32_t k, int K, const Fixed &ax) {
  uint64_t off = 0;
  for (int b = 0; b < K; ++b)
    if ((k >> b) & 1u) off |= 1ull << ax.pos[b];
  return off;
}

// Any K >= 6, complex128: out of place from `src` (a copy of the state) into
// psi, the product of the matrix and the 2^K x ngroups matrix of the groups.
// A workgroup takes 16 rows and CT blocks of 16 columns, its NW waves a share
// of the summed index each; their sums meet in LDS.  A wave's lanes
// take the summed index in fours (lane l: 4 (l / 16) .. + 3 of every 16), so
// that its matrix reads are 256-byte runs.  10 targets of 15 qubits (a 16 MiB
// matrix): 27 us with 16 waves on 16 columns, 44 with 4, 55 with 4 on 32
// columns, 904 with one thread per output; 10 targets of 22 qubits 0.7 ms
// besides the matrix's upload, was 17.6.  Errors against 80-bit products are
// a fifth to two thirds of those of one thread's chain (6 to 10 targets).
template <int CT, int NW>
__global__ __launch_bounds__(64 * NW) void k_dense_mm(double2 *__restrict__ psi,
                                                  const double2 *__restrict__ src,
                                                  uint64_t ngroups, int K, Fixed fx, Fixed ax,
                                                  const double2 *__restrict__ m) {
  __shared__ double2 part[NW][4][CT][64];
  const uint32_t D = 1u << K;
  const int tid = threadIdx.x, lane = tid & 63, c = lane & 15, q = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const uint64_t nrow = D / 16, ncol = (ngroups + 16 * CT - 1) / (16 * CT);
  const uint64_t oq = deposit(4u * q, K, ax);
  const uint64_t o1 = 1ull << ax.pos[0], o2 = 1ull << ax.pos[1];
  const uint32_t k0 = wave * (D / NW), k1 = k0 + D / NW;
  for (uint64_t tile = blockIdx.x; tile < nrow * ncol; tile += gridDim.x) {
    const uint32_t r0 = (uint32_t)(tile % nrow) * 16;
    const uint64_t g0 = (tile / nrow) * (16 * CT);
    const double2 *col[CT];
#pragma unroll
    for (int j = 0; j < CT; ++j) {
      const uint64_t g = g0 + 16 * j + c;  // past the last group: group 0, not stored
      col[j] = src + (expand(g < ngroups ? g : 0, fx) | oq);
    }
    const double2 *row = m + (uint64_t)(r0 + c) * D + 4 * q;
    CplxAcc acc[CT];
#pragma unroll
    for (int j = 0; j < CT; ++j) acc[j].clear();
#pragma unroll 2
    for (uint32_t k = k0; k < k1; k += 16) {
      const uint64_t ok = deposit(k, K, ax);
      double2 a[4], b[4][CT];
#pragma unroll
      for (int s = 0; s < 4; ++s) a[s] = row[k + s];
#pragma unroll
      for (int s = 0; s < 4; ++s)
#pragma unroll
        for (int j = 0; j < CT; ++j)
          b[s][j] = col[j][ok + ((s & 1) ? o1 : 0) + ((s & 2) ? o2 : 0)];
#pragma unroll
      for (int s = 0; s < 4; ++s)
#pragma unroll
        for (int j = 0; j < CT; ++j) mfma_cplx<false>(acc[j], a[s].x, a[s].y, b[s][j]);
    }
#pragma unroll
    for (int v = 0; v < 4; ++v)
#pragma unroll
      for (int j = 0; j < CT; ++j) part[wave][v][j][lane] = acc[j].at(v);
    __syncthreads();
    if (wave < 4) {  // rows 4 wave .. 4 wave + 3
      const uint64_t out = deposit(r0 + 4u * wave + q, K, ax);
#pragma unroll
      for (int j = 0; j < CT; ++j) {
        double2 s = part[0][wave][j][lane];
#pragma unroll
        for (int w = 1; w < NW; ++w) {
          s.x += part[w][wave][j][lane].x;
          s.y += part[w][wave][j][lane].y;
        }
        const uint64_t g = g0 + 16 * j + c;
        if (g < ngroups) psi[expand(g, fx) | out] = s;
      }
    }
    __syncthreads();
  }
}

// Any K >= 6, complex64: the same product with one chain of FMAs per output,
// in the order of the summed index.  A workgroup takes 16 NR rows and 16 NC
// columns in steps of 64 values of the index, a thread NR x NC outputs 16
// apart.  In place (src == psi) when the rows are all of the matrix's: they
// are stored after the only step has been read.  Bound by FP32 issue and LDS
// reads: 27 qubits, 6 targets 1.4-1.7 ms, 25-28 ms with one thread per output.
template <int NR, int NC>
__global__ __launch_bounds__(256) void k_dense_f32(float2 *psi, const float2 *src,
                                                   uint64_t ngroups, int K, Fixed fx, Fixed ax,
                                                   const float2 *__restrict__ m) {
  constexpr int TR = 16 * NR, TC = 16 * NC, KC = 64;
  __shared__ float2 sa[KC][TR + 1];
  __shared__ float2 sb[KC][TC];
  __shared__ uint64_t soff[KC], sbase[TC];
  const uint32_t D = 1u << K;
  const int tid = threadIdx.x, tx = tid & 15, ty = tid >> 4;
  const uint64_t nrow = D / TR, ncol = (ngroups + TC - 1) / TC;
  if (tid < KC) soff[tid] = deposit(tid, 6, ax);
  for (uint64_t tile = blockIdx.x; tile < nrow * ncol; tile += gridDim.x) {
    const uint32_t r0 = (uint32_t)(tile % nrow) * TR;
    const uint64_t g0 = (tile / nrow) * TC;
    if (tid < TC) sbase[tid] = expand(g0 + tid < ngroups ? g0 + tid : 0, fx);
    float2 acc[NR][NC];
#pragma unroll
    for (int i = 0; i < NR; ++i)
#pragma unroll
      for (int j = 0; j < NC; ++j) acc[i][j] = czero<float2>();
    for (uint32_t k0 = 0; k0 < D; k0 += KC) {
      __syncthreads();
      const uint64_t ok = deposit(k0, K, ax);
      for (int e = tid; e < TR * KC; e += 256)
        sa[e % KC][e / KC] = m[(uint64_t)(r0 + e / KC) * D + k0 + e % KC];
      for (int e = tid; e < TC * KC; e += 256)
        sb[e / TC][e % TC] = src[sbase[e % TC] | soff[e / TC] | ok];
      __syncthreads();
#pragma unroll 4
      for (int k = 0; k < KC; ++k) {
        float2 a[NR], b[NC];
#pragma unroll
        for (int i = 0; i < NR; ++i) a[i] = sa[k][ty + 16 * i];
#pragma unroll
        for (int j = 0; j < NC; ++j) b[j] = sb[k][tx + 16 * j];
#pragma unroll
        for (int i = 0; i < NR; ++i)
#pragma unroll
          for (int j = 0; j < NC; ++j) acc[i][j] = cmla(acc[i][j], a[i].x, a[i].y, b[j]);
      }
    }
#pragma unroll
    for (int i = 0; i < NR; ++i) {
      const uint64_t out = deposit(r0 + ty + 16 * i, K, ax);
#pragma unroll
      for (int j = 0; j < NC; ++j)
        if (g0 + tx + 16 * j < ngroups) psi[sbase[tx + 16 * j] | out] = acc[i][j];
    }
    __syncthreads();
  }
}

// Which kernel a dense gate on na >= 4 qubits takes, nfree index bits being
// neither its targets nor its controls; low: a fixed bit among the lowest 4;
// big: a streaming state; eight: eight_streams below.  Measured, complex128
// (us per gate with its upload):
//   5 qubits, 15-qubit state: tiles 10-11, k_gatek and its staged form 40;
//   24 qubits: 95 against 108 (free low bits) and 95-115 against 180; 27
//   qubits: 800-1020 against 1170 (low bits fixed), but 870-1040 against
//   780-800 of k_gatek's long runs (low bits free), which it keeps.
//   4 qubits, free low bits: 13 against 17 up to 19 qubits, 32 against 39 at
//   20; 18 either way at 21, 27-33 against 25-29 at 22, 44-55 against 42-48 at
//   23, 75-90 against 72-82 at 24, so k_gatek from 21 on.  Low bits fixed:
//   27-31 against 37-39 at 22, 42-51 against 53-57 at 23, 74-82 against 83-87
//   at 24; at 28 qubits 1580-1850 against 1460-1600, so streaming states keep
//   theirs.
//   6 qubits: 32 columns per tile from 20 qubits on (33 against 37 at 20, 67
//   against 74 at 22, 1200 against 1240 at 27), 16 below (24 against 26).
// Larger products take 32 columns per workgroup when that still fills the
// chip.  Complex64: 64 x 64 outputs per workgroup from 20 qubits on.
enum DenseForm { kDenseDirect, kDenseTile, kDenseTileSmall, kDenseWide, kDenseNarrow };

static DenseForm dense_form(bool c64, int na, int nfree, bool low, bool big, bool eight) {
  if (c64) {
    if (na <= 5) return kDenseDirect;
    return nfree >= 6 && na + nfree >= 20 ? kDenseWide : kDenseNarrow;
  }
  if (na == 4)
    return nfree >= 6 && !big && !eight && (low || nfree <= 16) ? kDenseTile : kDenseDirect;
  if (na == 5) return nfree >= 5 && (low || (!big && !eight)) ? kDenseTile : kDenseDirect;
  if (na == 6 && nfree >= 4) return nfree < 14 ? kDenseTileSmall : kDenseTile;
  return nfree >= 5 && na + nfree >= 17 ? kDenseWide : kDenseNarrow;
}

// Whether a tile's rows are 8 streams 4 MiB or more apart, each a run of a few
// KiB, of a state just the size of the last-level cache (2^24 amplitudes of
// complex128).  There, tiles take 91-96 us (4 qubits, low bits fixed; 5
// qubits, low bits free) and the kernels without tiles 85-91 (4 qubits) and
// 87-88; with 4 or 16 streams, or shorter runs, tiles are faster as elsewhere.
static bool eight_streams(int n, uint64_t active) {
  return n == 24 && __builtin_popcountll(active >> 18) == 3 && (active & 0x3FF00ull) == 0;
}

bool dense_needs_scratch(bool c64, int n, const Gate &g) {
  if (g.na <= 5) return false;
  const Fixed fx = make_fixed(g.cmask | active_mask(g), g.cval);
  const DenseForm f = dense_form(c64, g.na, n - fx.nf, false, false, false);
  if (c64) return !(g.na == 6 && f == kDenseWide);
  return f != kDenseTile && f != kDenseTileSmall;
}

static TileMap tile_map(const Fixed &fx, const Fixed &ax, int lc) {
  const uint64_t fixed = fx_mask(fx);
  TileMap tm{};
  int slot = 0, col = 0;
  for (int q = 0; q < 64; ++q) {
    int row = -1;
    for (int j = 0; j < ax.nf; ++j)
      if (ax.pos[j] == q) row = j;
    if (row < 0 && (((fixed >> q) & 1ull) || col == lc)) continue;
    if (row >= 0) tm.row[row] = (uint8_t)slot;
    else tm.col[col++] = (uint8_t)slot;
    tm.pa[slot++] = (uint8_t)q;
  }
  return tm;
}

template <int K, int LC>
static void launch_dense_tile(double2 *psi, int nfree, const Fixed &fx, const Fixed &ax, bool real,
                              bool big, const double2 *m, hipStream_t s) {
  const TileMap tm = tile_map(fx, ax, LC);
  const uint64_t ntiles = 1ull << (nfree - LC);
  constexpr uint64_t kPerCU = K + LC == 11 ? 4 : 8;
  const unsigned grid = (unsigned)std::min<uint64_t>(ntiles, 256 * kPerCU);
  nt_dispatch(big, [&](auto nt) {
    if (K <= 5 && real)
      hipLaunchKernelGGL((k_dense_tile<K, LC, K <= 5, decltype(nt)::value>), dim3(grid),
                         dim3(256), 0, s, psi, ntiles, fx, tm, m);
    else
      hipLaunchKernelGGL((k_dense_tile<K, LC, false, decltype(nt)::value>), dim3(grid), dim3(256),
                         0, s, psi, ntiles, fx, tm, m);
  });
}

// Calls f(integral_constant K, integral_constant real) for K = na in 3..5.
template <typename F>
static void gatek_dispatch(int na, bool real, F &&f) {
  using std::integral_constant;
  if (real) {
    if (na == 3) f(integral_constant<int, 3>{}, integral_constant<bool, true>{});
    else if (na == 4) f(integral_constant<int, 4>{}, integral_constant<bool, true>{});
    else f(integral_constant<int, 5>{}, integral_constant<bool, true>{});
  } else {
    if (na == 3) f(integral_constant<int, 3>{}, integral_constant<bool, false>{});
    else if (na == 4) f(integral_constant<int, 4>{}, integral_constant<bool, false>{});
    else f(integral_constant<int, 5>{}, integral_constant<bool, false>{});
  }
}

// d_mat layout: row-major D x D {re, im} in precision R.  `scratch` (2^n amplitudes) is needed
// where dense_needs_scratch says so.
template <typename R>
hipError_t launch_gate_dense(void *psi_v, int n, const Gate &g, void *d_mat, void *scratch,
                             hipStream_t s) {
  using T = typename V2<R>::T;
  T *psi = (T *)psi_v;
  const uint64_t amask = active_mask(g);
  const Fixed fx = make_fixed(g.cmask | amask, g.cval);
  const int nfree = n - fx.nf;
  const uint64_t nfreeN = 1ull << nfree;
  const bool big = streaming(n, sizeof(T));
  // pair partners closer than a 128-byte line: plain loads (see kStreamBytes)
  const auto near = [](int q) { return (sizeof(T) << q) < 128; };
  // QS_GATE1_LANE=0 keeps k_gate1 for every target qubit
  static const bool lane_form = [] {
    const char *v = std::getenv("QS_GATE1_LANE");
    return !(v && v[0] == '0');
  }();
  if (g.na == 1 && g.act[0] < 6 && n >= 6 && (g.cmask & 0x3Full) == 0 && lane_form) {
    // measured at 30 qubits, complex128, on qubit 0: four streams 32 chunks
    // apart per workgroup 5.28 ms, one run of 4 chunks per wave 5.92 ms,
    // k_gate1 6.28-6.54 ms.  States of fewer than 128 chunks take the one-run
    // order (the four-stream order needs chunk bits 5 and 6).
    constexpr int kItems = 4;
    constexpr int kStreams = 4;
    const Fixed fxc = make_fixed(g.cmask >> 6, g.cval >> 6);
    const uint64_t nchunks = 1ull << (n - 6 - fxc.nf);
    const bool streams = nchunks >= 128;
    const unsigned grid = streams ? (unsigned)(nchunks / (4 * kItems * kStreams))
                                  : grid_for(nchunks * 64, kBlock * kItems);
    const MatArg<R, 2> ma = to_matarg<R, 2>(g);
    nt_dispatch(big, [&](auto nt) {
      constexpr bool NT = decltype(nt)::value;
      auto go = [&](auto kk) {
        if (streams)
          hipLaunchKernelGGL((k_gate1_lane<R, decltype(kk)::value, kItems, NT, kStreams>),
                             dim3(grid), dim3(kBlock), 0, s, psi, nchunks, fxc, ma);
        else
          hipLaunchKernelGGL((k_gate1_lane<R, decltype(kk)::value, kItems, NT>), dim3(grid),
                             dim3(kBlock), 0, s, psi, nchunks, fxc, ma);
      };
      switch (g.act[0]) {
        case 0: go(std::integral_constant<int, 0>{}); break;
        case 1: go(std::integral_constant<int, 1>{}); break;
        case 2: go(std::integral_constant<int, 2>{}); break;
        case 3: go(std::integral_constant<int, 3>{}); break;
        case 4: go(std::integral_constant<int, 4>{}); break;
        default: go(std::integral_constant<int, 5>{}); break;
      }
    });
  } else if (g.na == 1) {
    constexpr int kItems = 4;
    // streaming complex128 states, target not on qubits 0..2: two pairs per
    // unit, the second xbit away; xbit is qubit 12 (64 KiB of amplitudes)
    // when free, else qubit 11.  Complex64 keeps one pair per unit: at 30
    // qubits the two forms measured within +-4% of each other, either way
    // depending on the target (wall time per gate, 2.57-3.01 ms).
    // QS_GATE1_STREAMS=0 keeps one pair per unit.
    static const bool streams_on = [] {
      const char *v = std::getenv("QS_GATE1_STREAMS");
      return !(v && v[0] == '0');
    }();
    const uint64_t used = g.cmask | amask;
    int xq = -1;
    if (sizeof(T) == 16 && big && !near(g.act[0]) && streams_on) {
      for (int q : {12, 11})
        if (xq < 0 && q < n && !((used >> q) & 1ull)) xq = q;
    }
    if (xq >= 0) {
      const Fixed fxx = make_fixed(used | (1ull << xq), g.cval);
      const uint64_t nunits = nfreeN >> 1;
      hipLaunchKernelGGL((k_gate1<R, kItems, true, 2>), dim3(grid_for(nunits, kBlock * kItems)),
                         dim3(kBlock), 0, s, psi, nunits, fxx, 1ull << g.act[0],
                         to_matarg<R, 2>(g), 1ull << xq);
    } else {
      nt_dispatch(big && !near(g.act[0]), [&](auto nt) {
        hipLaunchKernelGGL((k_gate1<R, kItems, decltype(nt)::value>),
                           dim3(grid_for(nfreeN, kBlock * kItems)), dim3(kBlock), 0, s, psi,
                           nfreeN, fx, 1ull << g.act[0], to_matarg<R, 2>(g), (uint64_t)0);
      });
    }
  } else if (g.na == 2) {
    constexpr int kItems = 2;
    nt_dispatch(big && !near(g.act[0]) && !near(g.act[1]), [&](auto nt) {
      hipLaunchKernelGGL((k_gate2<R, kItems, decltype(nt)::value>),
                         dim3(grid_for(nfreeN, kBlock * kItems)), dim3(kBlock), 0, s, psi, nfreeN,
                         fx, 1ull << g.act[0], 1ull << g.act[1], to_matarg<R, 4>(g));
    });
  } else if (g.na >= 3 && g.na <= 5) {
    const Fixed ax = active_positions(g);
    const R *m = (const R *)d_mat;  // row-major {re, im}
    bool real = true;
    for (const cd &v : g.m) real = real && v.im == 0.0;
    if constexpr (std::is_same<R, double>::value) {
      if (g.na >= 4 &&
          dense_form(false, g.na, nfree, (fx_mask(fx) & 0xFull) != 0, big,
                     eight_streams(n, active_mask(g))) == kDenseTile) {
        if (g.na == 4)
          launch_dense_tile<4, 6>(psi, nfree, fx, ax, real, big, (const double2 *)m, s);
        else
          launch_dense_tile<5, 5>(psi, nfree, fx, ax, real, big, (const double2 *)m, s);
        return hipGetLastError();
      }
    }
    StageMap sm{};
    // fixed low bits (active or control on qubits 0..3) break the direct
    // kernel's 64-amplitude runs: stage through LDS instead
    if ((fx_mask(fx) & 0xFull) && stage_map(fx, ax, n, sm)) {
      const unsigned sgrid = (unsigned)(nfreeN / 64);
      auto staged = [&](auto kk, auto rr) {
        nt_dispatch(big, [&](auto nt) {
          // (complex128 blocks of 5 qubits on low bits are tiles)
          if constexpr (!(std::is_same<R, double>::value && decltype(kk)::value == 5))
            hipLaunchKernelGGL((k_gatek_staged<R, decltype(kk)::value, decltype(rr)::value,
                                               decltype(nt)::value>),
                               dim3(sgrid), dim3(64), 0, s, psi, nfreeN, fx, sm, m);
        });
      };
      gatek_dispatch(g.na, real, staged);
      return hipGetLastError();
    }
    if constexpr (std::is_same<R, float>::value) {
      // the matrix cores when the lowest 6 (or 5) index bits are free
      const uint64_t low = fx_mask(fx);
      if (g.na == 5 && !real && gatek_mfma() && (low & 0x1Full) == 0 && nfreeN % 64 == 0) {
        const bool wide = (low & 0x20ull) == 0;
        const uint64_t nchunks = nfreeN / (wide ? 64 : 32);
        const unsigned mgrid = (unsigned)std::min<uint64_t>(nchunks, 8192);
        nt_dispatch(big, [&](auto nt) {
          if (wide)
            hipLaunchKernelGGL((k_gatek5_mfma<decltype(nt)::value>), dim3(mgrid), dim3(64), 0,
                               s, (float2 *)psi, nchunks, fx, ax, (const float *)m);
          else
            hipLaunchKernelGGL((k_gatek5_mfma32<decltype(nt)::value>), dim3(mgrid), dim3(64), 0,
                               s, (float2 *)psi, nchunks, fx, ax, (const float *)m);
        });
        return hipGetLastError();
      }
    }
    const unsigned grid = grid_for(nfreeN, kBlock);
    auto direct = [&](auto kk, auto rr) {
      nt_dispatch(big, [&](auto nt) {
        hipLaunchKernelGGL((k_gatek<R, decltype(kk)::value, decltype(rr)::value,
                                    decltype(nt)::value>),
                           dim3(grid), dim3(kBlock), 0, s, psi, nfreeN, fx, ax, m);
      });
    };
    gatek_dispatch(g.na, real, direct);
  } else {
    const Fixed ax = active_positions(g);
    const T *m = (const T *)d_mat;
    const DenseForm f = dense_form(std::is_same<R, float>::value, g.na, nfree, false, big, false);
    const T *src = psi;
    if (dense_needs_scratch(std::is_same<R, float>::value, n, g)) {
      hipError_t e = hipMemcpyAsync(scratch, psi, sizeof(T) << n, hipMemcpyDeviceToDevice, s);
      if (e != hipSuccess) return e;
      src = (const T *)scratch;
    }
    const auto grid = [&](uint64_t rows, uint64_t cols) {
      return dim3((unsigned)std::min<uint64_t>(
          ((1ull << g.na) / rows) * ((nfreeN + cols - 1) / cols), 65536));
    };
    if constexpr (std::is_same<R, double>::value) {
      if (f == kDenseTile)
        launch_dense_tile<6, 5>(psi, nfree, fx, ax, false, big, m, s);
      else if (f == kDenseTileSmall)
        launch_dense_tile<6, 4>(psi, nfree, fx, ax, false, big, m, s);
      else if (f == kDenseWide)
        hipLaunchKernelGGL((k_dense_mm<2, 4>), grid(16, 32), dim3(256), 0, s, psi, src, nfreeN,
                           g.na, fx, ax, m);
      else if (g.na >= 8)  // a share is at least 16 of the 2^na values
        hipLaunchKernelGGL((k_dense_mm<1, 16>), grid(16, 16), dim3(1024), 0, s, psi, src, nfreeN,
                           g.na, fx, ax, m);
      else
        hipLaunchKernelGGL((k_dense_mm<1, 4>), grid(16, 16), dim3(256), 0, s, psi, src, nfreeN,
                           g.na, fx, ax, m);
    } else {
      if (f == kDenseWide)
        hipLaunchKernelGGL((k_dense_f32<4, 4>), grid(64, 64), dim3(256), 0, s, psi, src, nfreeN,
                           g.na, fx, ax, m);
      else
        hipLaunchKernelGGL((k_dense_f32<1, 1>), grid(16, 16), dim3(256), 0, s, psi, src, nfreeN,
                           g.na, fx, ax, m);
    }
  }
  return hipGetLastError();
}

// ---- permutation gates ------------------------------------------------------------

// Monomial gate (kPerm) out of place: every amplitude idx of the controlled
// subspace, with act pattern r, becomes ph[r] * src[idx with act pattern
// perm[r]].  `src` is a copy of the state; amplitudes outside the
// controlled subspace are left as they are.  Two passes over the state (the
// copy and the gather) whatever the arity, against 2^na complex products
// per amplitude for the dense form.
template <typename R>
__global__ __launch_bounds__(kBlock) void k_perm(typename V2<R>::T *__restrict__ psi,
                                                 const typename V2<R>::T *__restrict__ src,
                                                 uint64_t count, Fixed cx, Fixed ax,
                                                 const uint32_t *__restrict__ perm,
                                                 const typename V2<R>::T *__restrict__ ph) {
  using T = typename V2<R>::T;
  uint64_t amask = 0;
  for (int j = 0; j < ax.nf; ++j) amask |= 1ull << ax.pos[j];
  for (uint64_t p = (uint64_t)blockIdx.x * kBlock + threadIdx.x; p < count;
       p += (uint64_t)gridDim.x * kBlock) {
    const uint64_t idx = expand(p, cx);
    uint32_t r = 0;
    for (int j = 0; j < ax.nf; ++j) r |= (uint32_t)((idx >> ax.pos[j]) & 1ull) << j;
    const uint32_t c = perm[r];
    uint64_t sidx = idx & ~amask;
    for (int j = 0; j < ax.nf; ++j)
      if ((c >> j) & 1u) sidx |= 1ull << ax.pos[j];
    const T f = ph[r];
    psi[idx] = cmla(czero<T>(), f.x, f.y, src[sidx]);
  }
}

size_t perm_table_phase_offset(int na) { return ((sizeof(uint32_t) << na) + 15) & ~(size_t)15; }

template <typename R>
hipError_t launch_gate_perm(void *psi, int n, const Gate &g, const void *d_tab, void *scratch,
                            hipStream_t s) {
  using T = typename V2<R>::T;
  const Fixed cx = make_fixed(g.cmask, g.cval);
  const Fixed ax = active_positions(g);
  hipError_t e = hipMemcpyAsync(scratch, psi, sizeof(T) << n, hipMemcpyDeviceToDevice, s);
  if (e != hipSuccess) return e;
  const uint64_t count = 1ull << (n - cx.nf);
  unsigned grid = grid_for(count, kBlock * 4);
  if (grid > 262144) grid = 262144;
  const char *tab = (const char *)d_tab;
  hipLaunchKernelGGL(k_perm<R>, dim3(grid), dim3(kBlock), 0, s, (T *)psi, (const T *)scratch,
                     count, cx, ax, (const uint32_t *)tab,
                     (const T *)(tab + perm_table_phase_offset(g.na)));
  return hipGetLastError();
}

// ---- diagonal gates -------------------------------------------------------------

// Multiply every amplitude whose control bits match by d[pattern of act bits].
template <typename R, bool kNT>
__global__ __launch_bounds__(kBlock) void k_diag(typename V2<R>::T *__restrict__ psi,
                                                 uint64_t count, Fixed cx, Fixed ax,
                                                 const typename V2<R>::T *__restrict__ d) {
  using T = typename V2<R>::T;
  for (uint64_t p = (uint64_t)blockIdx.x * kBlock + threadIdx.x; p < count;
       p += (uint64_t)gridDim.x * kBlock) {
    const uint64_t idx = expand(p, cx);
    uint32_t pat = 0;
    for (int j = 0; j < ax.nf; ++j) pat |= (uint32_t)((idx >> ax.pos[j]) & 1ull) << j;
    const T dv = d[pat];
    T a = ld<kNT>(psi + idx);
    T r = czero<T>();
    r = cmla(r, dv.x, dv.y, a);
    st<kNT>(psi + idx, r);
  }
}

template <typename R>
hipError_t launch_gate_diag(void *psi, int n, const Gate &g, void *d_mat, hipStream_t s) {
  using T = typename V2<R>::T;
  const Fixed cx = make_fixed(g.cmask, g.cval);
  const Fixed ax = active_positions(g);
  const uint64_t count = 1ull << (n - cx.nf);
  unsigned grid = grid_for(count, kBlock * 4);
  if (grid > 262144) grid = 262144;
  nt_dispatch(streaming(n, sizeof(T)), [&](auto nt) {
    hipLaunchKernelGGL((k_diag<R, decltype(nt)::value>), dim3(grid), dim3(kBlock), 0, s, (T *)psi,
                       count, cx, ax, (const T *)d_mat);
  });
  return hipGetLastError();
}

// Up to kMaxSparse (pattern, value) exceptions of a diagonal that is 1
// elsewhere.
constexpr int kMaxSparse = 16;
template <typename R>
struct SparseArg {
  uint64_t pat[kMaxSparse];
  R re[kMaxSparse], im[kMaxSparse];
  int count;
};

template <typename R, bool kNT>
__global__ __launch_bounds__(kBlock) void k_sparse(typename V2<R>::T *__restrict__ psi,
                                                   uint64_t per, Fixed fx, SparseArg<R> sp) {
  using T = typename V2<R>::T;
  const uint64_t total = per * (uint64_t)sp.count;
  for (uint64_t w = (uint64_t)blockIdx.x * kBlock + threadIdx.x; w < total;
       w += (uint64_t)gridDim.x * kBlock) {
    const uint64_t e = w / per, p = w % per;
    const uint64_t idx = expand(p, fx) | sp.pat[e];
    T a = ld<kNT>(psi + idx);
    T r = czero<T>();
    r = cmla(r, sp.re[e], sp.im[e], a);
    st<kNT>(psi + idx, r);
  }
}

template <typename R>
hipError_t launch_gate_sparse(void *psi, int n, const Gate &g, hipStream_t s) {
  using T = typename V2<R>::T;
  SparseArg<R> sp{};
  sp.count = (int)g.spat.size();
  if (sp.count > kMaxSparse) return hipErrorInvalidValue;
  if (sp.count == 0) return hipSuccess;
  for (int e = 0; e < sp.count; ++e) {
    sp.pat[e] = g.spat[e];
    sp.re[e] = (R)g.m[e].re;
    sp.im[e] = (R)g.m[e].im;
  }
  const Fixed fx = make_fixed(g.smask, 0);
  const uint64_t per = 1ull << (n - fx.nf);
  unsigned grid = grid_for(per * sp.count, kBlock * 4);
  if (grid > 262144) grid = 262144;
  nt_dispatch(streaming(n, sizeof(T)), [&](auto nt) {
    hipLaunchKernelGGL((k_sparse<R, decltype(nt)::value>), dim3(grid), dim3(kBlock), 0, s,
                       (T *)psi, per, fx, sp);
  });
  return hipGetLastError();
}

// ---- reductions -------------------------------------------------------------------

template <int N>
__device__ __forceinline__ void block_sum(double (&v)[N], double (*sh)[kBlock]) {
#pragma unroll
  for (int c = 0; c < N; ++c) sh[c][threadIdx.x] = v[c];
  __syncthreads();
  for (int w = kBlock / 2; w > 0; w >>= 1) {
    if ((int)threadIdx.x < w) {
#pragma unroll
      for (int c = 0; c < N; ++c) sh[c][threadIdx.x] += sh[c][threadIdx.x + w];
    }
    __syncthreads();
  }
#pragma unroll
  for (int c = 0; c < N; ++c) v[c] = sh[c][0];
}

// Second stage: one block sums nblocks partials of N channels (fixed order).
template <int N>
__global__ __launch_bounds__(kBlock) void k_finish(const double *__restrict__ part, int nblocks,
                                                   double *__restrict__ out) {
  __shared__ double sh[N][kBlock];
  double v[N];
#pragma unroll
  for (int c = 0; c < N; ++c) v[c] = 0.0;
  for (int b = threadIdx.x; b < nblocks; b += kBlock)
#pragma unroll
    for (int c = 0; c < N; ++c) v[c] += part[(size_t)b * N + c];
  block_sum<N>(v, sh);
  if (threadIdx.x == 0)
#pragma unroll
    for (int c = 0; c < N; ++c) out[c] = v[c];
}

static inline int reduce_grid(uint64_t len) {
  uint64_t g = (len + kBlock - 1) / kBlock;
  if (g > (uint64_t)kReduceBlocks) g = kReduceBlocks;
  if (g < 1) g = 1;
  return (int)g;
}

// Block order of the reductions over a state of at least kReduceBlocks *
// kRedTrip amplitudes: block b owns the len / gridDim.x consecutive
// amplitudes from b * len / gridDim.x and reads them in trips of kRedTrip
// (a contiguous 64 KiB of complex128, 16 nontemporal loads in flight per
// thread); each thread adds its amplitudes in index order.  Smaller states
// take the grid-stride order.  Measured at 2^30 complex128 amplitudes, read
// and split by one bit: 2.42-2.45 ms (0.88 of 8 TB/s) against 3.07 ms for the
// grid-stride order with four ordinary loads in flight (2.92 ms nontemporal).
constexpr int kRedLoads = 16;
constexpr uint64_t kRedTrip = (uint64_t)kRedLoads * kBlock;

static inline bool reduce_blocked(uint64_t len) {
  return len >= (uint64_t)kReduceBlocks * kRedTrip;
}

// What becomes of a split's sums: {prob_0, prob_1} go to `host`, or, with a
// slot, the outcome is decided here (src/register.rs:317-321: x > prob_0),
// stored there and left with its scale in `coll` for the collapse.
__device__ __forceinline__ void split_result(const double (&v)[2], const SplitEnd &end) {
  if (threadIdx.x != 0) return;
  if (end.host) {
    end.host[0] = v[0];
    end.host[1] = v[1];
  }
  if (end.slot) {
    const int res = end.x > v[0];
    end.coll[0] = (double)res;
    end.coll[1] = sqrt(res ? v[1] : v[0]);
    *end.slot = (unsigned char)res;
  }
}

// The end of a split over all blocks: the partials go to `part`, and the
// block that comes last (it counts them, and leaves the counter at 0) adds
// them up in the order of k_finish.  Without a counter, k_split_finish does.
// Returns whether this block was the last; v holds the sums on its threads.
__device__ __forceinline__ bool split_end(double (&v)[2], double (*sh)[kBlock],
                                          double *__restrict__ part, const SplitEnd &end) {
  __shared__ bool last;
  if (gridDim.x > 1) {
    if (!end.count) {
      if (threadIdx.x == 0)
        for (int c = 0; c < 2; ++c) part[2 * blockIdx.x + c] = v[c];
      return false;
    }
    if (threadIdx.x == 0) {
      for (int c = 0; c < 2; ++c)
        __hip_atomic_store(part + 2 * blockIdx.x + c, v[c], __ATOMIC_RELAXED,
                           __HIP_MEMORY_SCOPE_AGENT);
      last = __hip_atomic_fetch_add(end.count, 1u, __ATOMIC_ACQ_REL, __HIP_MEMORY_SCOPE_AGENT) ==
             gridDim.x - 1;
    }
    __syncthreads();
    if (!last) return false;
    v[0] = v[1] = 0.0;
    for (unsigned b = threadIdx.x; b < gridDim.x; b += kBlock)
      for (int c = 0; c < 2; ++c)
        v[c] += __hip_atomic_load(part + 2 * b + c, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    block_sum<2>(v, sh);
    if (threadIdx.x == 0)
      __hip_atomic_store(end.count, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
  split_result(v, end);
  return true;
}

__global__ __launch_bounds__(kBlock) void k_split_finish(const double *__restrict__ part, int nblocks,
                                                         SplitEnd end) {
  __shared__ double sh[2][kBlock];
  double v[2] = {0.0, 0.0};
  for (int b = threadIdx.x; b < nblocks; b += kBlock)
    for (int c = 0; c < 2; ++c) v[c] += part[2 * b + c];
  block_sum<2>(v, sh);
  split_result(v, end);
}

// Grids up to which the last block takes the sums itself: each block's count
// is an atomic and a write-back of its XCD's L2, which a large grid pays for
// hundreds of times.  Twelve measures, complex128: 14 qubits (64 blocks) 197
// us in one launch each, 213 in two and a copy to the host; 15 qubits 213 us,
// 198 in two launches (this kernel writes to the host); 18 qubits 463, 214;
// 22 qubits 894, 417.  A deferred measure of up to 8 qubits is one launch of
// 2.4 us with its collapse, in four it was 6.6.
constexpr int kSplitBlocks = 64;

// Runs a split of g blocks, launch(end) being its kernel.
template <typename F>
static hipError_t run_split(int g, const SplitEnd &end, const double *d_part, hipStream_t s,
                            F &&launch) {
  SplitEnd mine = end;
  if (g > kSplitBlocks) mine.count = nullptr;
  launch(mine);
  if (g > kSplitBlocks)
    hipLaunchKernelGGL(k_split_finish, dim3(1), dim3(kBlock), 0, s, d_part, g, end);
  return hipGetLastError();
}

// Amplitude a of index i after a collapse on bit `target` of outcome `keep`.
template <typename R, typename T>
__device__ __forceinline__ T collapsed(T a, uint64_t i, int target, int keep, double sq) {
  if ((int)((i >> target) & 1ull) != keep) return czero<T>();
  a.x = (R)((double)a.x / sq);
  a.y = (R)((double)a.y / sq);
  return a;
}

template <typename R, bool kBlocked>
__global__ __launch_bounds__(kBlock) void k_prob_split(typename V2<R>::T *__restrict__ psi,
                                                       uint64_t len, int target,
                                                       double *__restrict__ part, SplitEnd end) {
  __shared__ double sh[2][kBlock];
  double v[2] = {0.0, 0.0};
  // each thread adds its amplitudes in index order (k_collapse_split relies
  // on the same order)
  if constexpr (kBlocked) {
    const uint64_t per = len / gridDim.x;
    const uint64_t b0 = (uint64_t)blockIdx.x * per + threadIdx.x;
    for (uint64_t w = b0; w < b0 + per; w += kRedTrip) {
      typename V2<R>::T a[kRedLoads];
#pragma unroll
      for (int k = 0; k < kRedLoads; ++k) a[k] = ld<true>(psi + w + (uint64_t)k * kBlock);
#pragma unroll
      for (int k = 0; k < kRedLoads; ++k) {
        const double re = (double)a[k].x, im = (double)a[k].y;
        const double p = re * re + im * im;
        if (((w + (uint64_t)k * kBlock) >> target) & 1ull)
          v[1] += p;
        else
          v[0] += p;
      }
    }
    block_sum<2>(v, sh);
    split_end(v, sh, part, end);
    return;
  }
  // four loads in flight per trip
  const uint64_t S = (uint64_t)gridDim.x * kBlock;
  uint64_t i = (uint64_t)blockIdx.x * kBlock + threadIdx.x;
  for (; i + 3 * S < len; i += 4 * S) {
    typename V2<R>::T a[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) a[k] = psi[i + k * S];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const double re = (double)a[k].x, im = (double)a[k].y;
      const double p = re * re + im * im;
      if (((i + k * S) >> target) & 1ull)
        v[1] += p;
      else
        v[0] += p;
    }
  }
  for (; i < len; i += S) {
    const auto a = psi[i];
    const double re = (double)a.x, im = (double)a.y;
    const double p = re * re + im * im;
    if ((i >> target) & 1ull)
      v[1] += p;
    else
      v[0] += p;
  }
  block_sum<2>(v, sh);
  split_end(v, sh, part, end);
  if (end.slot && gridDim.x == 1) {  // one block: the collapse as well
    const int keep = end.x > v[0];
    const double sq = sqrt(keep ? v[1] : v[0]);
    for (i = threadIdx.x; i < len; i += kBlock)
      psi[i] = collapsed<R>(psi[i], i, target, keep, sq);
  }
}

template <typename R>
hipError_t launch_prob_split(void *psi, int n, int target, double *d_part, const SplitEnd &end,
                             hipStream_t s) {
  const uint64_t len = 1ull << n;
  const int g = reduce_grid(len);
  return run_split(g, end, d_part, s, [&](const SplitEnd &e) {
    if (reduce_blocked(len))
      hipLaunchKernelGGL((k_prob_split<R, true>), dim3(g), dim3(kBlock), 0, s,
                         (typename V2<R>::T *)psi, len, target, d_part, e);
    else
      hipLaunchKernelGGL((k_prob_split<R, false>), dim3(g), dim3(kBlock), 0, s,
                         (typename V2<R>::T *)psi, len, target, d_part, e);
  });
}

// The collapse of try_measure (src/register.rs:324-339): zero the amplitudes
// whose target bit differs from the outcome; divide the rest, component by
// component, by sqrt(total).
template <typename R>
__global__ __launch_bounds__(kBlock) void k_collapse(typename V2<R>::T *__restrict__ psi,
                                                     uint64_t len, int target, int keep,
                                                     double sq) {
  for (uint64_t i = (uint64_t)blockIdx.x * kBlock + threadIdx.x; i < len;
       i += (uint64_t)gridDim.x * kBlock) {
    psi[i] = collapsed<R>(psi[i], i, target, keep, sq);
  }
}

// The collapse of one measure fused with the probability split of the next
// (src/register.rs:297-339 twice): amplitudes whose bit `ctarget` differs
// from `keep` are zeroed, the rest divided by sqrt(total), and the squared
// moduli of the values stored (after rounding to R) are summed by bit
// `target`, over the same grid, in the same order and with the same block
// sums as k_prob_split on the collapsed state, so {prob_0, prob_1} are the
// same bits as a separate split would give.  One pass instead of two: the
// split's full read of the collapsed state is saved.
template <typename R, bool kBlocked>
__global__ __launch_bounds__(kBlock) void k_collapse_split(typename V2<R>::T *__restrict__ psi,
                                                           uint64_t len, int ctarget, int keep,
                                                           double sq, int target,
                                                           double *__restrict__ part,
                                                           SplitEnd end) {
  using T = typename V2<R>::T;
  __shared__ double sh[2][kBlock];
  double v[2] = {0.0, 0.0};
  auto one = [&](uint64_t i, T a) {
    a = collapsed<R>(a, i, ctarget, keep, sq);
    st<kBlocked>(psi + i, a);
    const double re = (double)a.x, im = (double)a.y;
    const double p = re * re + im * im;
    if ((i >> target) & 1ull)
      v[1] += p;
    else
      v[0] += p;
  };
  // the trip structure and order of k_prob_split; only kept amplitudes are
  // read
  if constexpr (kBlocked) {
    const uint64_t per = len / gridDim.x;
    const uint64_t b0 = (uint64_t)blockIdx.x * per + threadIdx.x;
    for (uint64_t w = b0; w < b0 + per; w += kRedTrip) {
      T a[kRedLoads];
#pragma unroll
      for (int k = 0; k < kRedLoads; ++k) {
        const uint64_t i = w + (uint64_t)k * kBlock;
        a[k] = (int)((i >> ctarget) & 1ull) == keep ? ld<true>(psi + i) : czero<T>();
      }
#pragma unroll
      for (int k = 0; k < kRedLoads; ++k) one(w + (uint64_t)k * kBlock, a[k]);
    }
    block_sum<2>(v, sh);
    split_end(v, sh, part, end);
    return;
  }
  const uint64_t S = (uint64_t)gridDim.x * kBlock;
  uint64_t i = (uint64_t)blockIdx.x * kBlock + threadIdx.x;
  for (; i + 3 * S < len; i += 4 * S) {
    T a[4];
#pragma unroll
    for (int k = 0; k < 4; ++k)
      a[k] = (int)(((i + k * S) >> ctarget) & 1ull) == keep ? psi[i + k * S] : czero<T>();
#pragma unroll
    for (int k = 0; k < 4; ++k) one(i + k * S, a[k]);
  }
  for (; i < len; i += S) one(i, (int)((i >> ctarget) & 1ull) == keep ? psi[i] : czero<T>());
  block_sum<2>(v, sh);
  split_end(v, sh, part, end);
}

template <typename R>
hipError_t launch_collapse_split(void *psi, int n, int ctarget, int keep, double total,
                                 int target, double *d_part, const SplitEnd &end, hipStream_t s) {
  const uint64_t len = 1ull << n;
  const int g = reduce_grid(len);
  return run_split(g, end, d_part, s, [&](const SplitEnd &e) {
    if (reduce_blocked(len))
      hipLaunchKernelGGL((k_collapse_split<R, true>), dim3(g), dim3(kBlock), 0, s,
                         (typename V2<R>::T *)psi, len, ctarget, keep, sqrt(total), target, d_part,
                         e);
    else
      hipLaunchKernelGGL((k_collapse_split<R, false>), dim3(g), dim3(kBlock), 0, s,
                         (typename V2<R>::T *)psi, len, ctarget, keep, sqrt(total), target, d_part,
                         e);
  });
}

// k_collapse with its outcome and scale read from device memory.
template <typename R>
__global__ __launch_bounds__(kBlock) void k_collapse_dev(typename V2<R>::T *__restrict__ psi,
                                                         uint64_t len, int target,
                                                         const double *__restrict__ coll) {
  const int keep = (int)coll[0];
  const double sq = coll[1];
  for (uint64_t i = (uint64_t)blockIdx.x * kBlock + threadIdx.x; i < len;
       i += (uint64_t)gridDim.x * kBlock) {
    psi[i] = collapsed<R>(psi[i], i, target, keep, sq);
  }
}

template <typename R>
hipError_t launch_measure_deferred(void *psi, int n, int target, double x, double *d_part,
                                   double *d_coll, unsigned *d_count, unsigned char *d_slot,
                                   hipStream_t s) {
  const uint64_t len = 1ull << n;
  SplitEnd end;
  end.count = d_count;
  end.x = x;
  end.coll = d_coll;
  end.slot = d_slot;
  hipError_t e = launch_prob_split<R>(psi, n, target, d_part, end, s);
  if (e != hipSuccess || reduce_grid(len) == 1) return e;
  unsigned grid = grid_for(len, kBlock * 4);
  if (grid > 262144) grid = 262144;
  hipLaunchKernelGGL(k_collapse_dev<R>, dim3(grid), dim3(kBlock), 0, s, (typename V2<R>::T *)psi,
                     len, target, (const double *)d_coll);
  return hipGetLastError();
}

// The collapse onto the amplitudes i with (i & mask) == pat (k_collapse:
// one target bit; the mask collapse of measure_sequence: every decided
// qubit), over chunks of 64 amplitudes in the stream order of k_gate1_lane
// (four streams 32 chunks apart per workgroup, 16 chunks per workgroup per
// stream); lane l takes amplitude l of each chunk, reads it only when it is
// kept.  nchunks is a power of two >= 128; the host launches
// nchunks / 64 workgroups.  Measured at 30 qubits, complex128, collapse on
// qubit 29 (half the state read, all of it written): 4.08 ms (6.3 TB/s)
// against 4.78 ms for the grid-stride k_collapse.
template <typename R>
__global__ __launch_bounds__(kBlock) void k_collapse_streams(typename V2<R>::T *__restrict__ psi,
                                                             uint64_t nchunks, uint64_t mask,
                                                             uint64_t pat, double sq) {
  using T = typename V2<R>::T;
  constexpr int kItems = 4, S = 4;
  if (((uint64_t)blockIdx.x + 1) * (4 * kItems * S) > nchunks) return;
  const uint64_t lane = threadIdx.x & 63;
  uint64_t idx[kItems * S];
  T a[kItems * S];
#pragma unroll
  for (int it = 0; it < kItems; ++it) {
    const uint64_t u = (uint64_t)blockIdx.x * (4 * kItems) + it * 4 + (threadIdx.x >> 6);
    const uint64_t c0 = (u & 31ull) | ((u >> 5) << 7);
#pragma unroll
    for (int st_ = 0; st_ < S; ++st_) idx[it * S + st_] = ((c0 | ((uint64_t)st_ << 5)) << 6) | lane;
  }
#pragma unroll
  for (int j = 0; j < kItems * S; ++j)
    a[j] = (idx[j] & mask) == pat ? ld<true>(psi + idx[j]) : czero<T>();
#pragma unroll
  for (int j = 0; j < kItems * S; ++j) {
    T r = a[j];
    r.x = (R)((double)r.x / sq);
    r.y = (R)((double)r.y / sq);
    st<true>(psi + idx[j], r);
  }
}

template <typename R>
hipError_t launch_collapse_pattern(void *psi, int n, uint64_t mask, uint64_t pat, double total,
                                   hipStream_t s) {
  const uint64_t nchunks = (1ull << n) >> 6;
  if (n < 13) return hipErrorInvalidValue;  // the stream order needs 128 chunks
  hipLaunchKernelGGL(k_collapse_streams<R>, dim3((unsigned)(nchunks / 64)), dim3(kBlock), 0, s,
                     (typename V2<R>::T *)psi, nchunks, mask, pat, sqrt(total));
  return hipGetLastError();
}

template <typename R>
hipError_t launch_collapse(void *psi, int n, int target, int keep, double total, hipStream_t s) {
  const uint64_t len = 1ull << n;
  if (streaming(n, sizeof(typename V2<R>::T))) {
    // states above the last-level cache: the stream order
    return launch_collapse_pattern<R>(psi, n, 1ull << target, (uint64_t)keep << target, total, s);
  }
  unsigned grid = grid_for(len, kBlock * 4);
  if (grid > 262144) grid = 262144;
  hipLaunchKernelGGL(k_collapse<R>, dim3(grid), dim3(kBlock), 0, s, (typename V2<R>::T *)psi, len,
                     target, keep, sqrt(total));
  return hipGetLastError();
}

template <typename R, bool kBlocked>
__global__ __launch_bounds__(kBlock) void k_norm(const typename V2<R>::T *__restrict__ psi,
                                                 uint64_t len, double *__restrict__ part) {
  __shared__ double sh[1][kBlock];
  double v[1] = {0.0};
  if constexpr (kBlocked) {
    const uint64_t per = len / gridDim.x;
    const uint64_t b0 = (uint64_t)blockIdx.x * per + threadIdx.x;
    for (uint64_t w = b0; w < b0 + per; w += kRedTrip) {
      typename V2<R>::T a[kRedLoads];
#pragma unroll
      for (int k = 0; k < kRedLoads; ++k) a[k] = ld<true>(psi + w + (uint64_t)k * kBlock);
#pragma unroll
      for (int k = 0; k < kRedLoads; ++k)
        v[0] += (double)a[k].x * (double)a[k].x + (double)a[k].y * (double)a[k].y;
    }
  } else {
    for (uint64_t i = (uint64_t)blockIdx.x * kBlock + threadIdx.x; i < len;
         i += (uint64_t)gridDim.x * kBlock) {
      const auto a = psi[i];
      v[0] += (double)a.x * (double)a.x + (double)a.y * (double)a.y;
    }
  }
  block_sum<1>(v, sh);
  if (threadIdx.x == 0) part[blockIdx.x] = v[0];
}

template <typename R>
hipError_t launch_norm(const void *psi, int n, double *d_part, double *d_out, hipStream_t s) {
  const uint64_t len = 1ull << n;
  const int g = reduce_grid(len);
  if (reduce_blocked(len))
    hipLaunchKernelGGL((k_norm<R, true>), dim3(g), dim3(kBlock), 0, s,
                       (const typename V2<R>::T *)psi, len, d_part);
  else
    hipLaunchKernelGGL((k_norm<R, false>), dim3(g), dim3(kBlock), 0, s,
                       (const typename V2<R>::T *)psi, len, d_part);
  hipLaunchKernelGGL(k_finish<1>, dim3(1), dim3(kBlock), 0, s, (const double *)d_part, g, d_out);
  return hipGetLastError();
}

template <typename Ra, typename Rb>
__global__ __launch_bounds__(kBlock) void k_inner(const typename V2<Ra>::T *__restrict__ a,
                                                  const typename V2<Rb>::T *__restrict__ b,
                                                  uint64_t len, double *__restrict__ part) {
  __shared__ double sh[2][kBlock];
  double v[2] = {0.0, 0.0};
  for (uint64_t i = (uint64_t)blockIdx.x * kBlock + threadIdx.x; i < len;
       i += (uint64_t)gridDim.x * kBlock) {
    const auto x = a[i];
    const auto y = b[i];
    const double xr = x.x, xi = x.y, yr = y.x, yi = y.y;
    v[0] += xr * yr + xi * yi;  // Re conj(x) y
    v[1] += xr * yi - xi * yr;  // Im conj(x) y
  }
  block_sum<2>(v, sh);
  if (threadIdx.x == 0) {
    part[2 * blockIdx.x] = v[0];
    part[2 * blockIdx.x + 1] = v[1];
  }
}

template <typename Ra, typename Rb>
static void inner_launch(const void *a, const void *b, uint64_t len, int g, double *d_part,
                         hipStream_t s) {
  hipLaunchKernelGGL((k_inner<Ra, Rb>), dim3(g), dim3(kBlock), 0, s,
                     (const typename V2<Ra>::T *)a, (const typename V2<Rb>::T *)b, len, d_part);
}

hipError_t launch_inner(const void *a, bool a_c64, const void *b, bool b_c64, int n,
                        double *d_part, double *d_out, hipStream_t s) {
  const uint64_t len = 1ull << n;
  const int g = reduce_grid(len);
  if (!a_c64 && !b_c64) inner_launch<double, double>(a, b, len, g, d_part, s);
  if (!a_c64 && b_c64) inner_launch<double, float>(a, b, len, g, d_part, s);
  if (a_c64 && !b_c64) inner_launch<float, double>(a, b, len, g, d_part, s);
  if (a_c64 && b_c64) inner_launch<float, float>(a, b, len, g, d_part, s);
  hipLaunchKernelGGL(k_finish<2>, dim3(1), dim3(kBlock), 0, s, (const double *)d_part, g, d_out);
  return hipGetLastError();
}

// Count of amplitudes where !(|a_i - b_i| < tol) -- NaN counts as unequal,
// as `e.norm() < 1e-8` is false for NaN in PartialEq (src/register.rs:411).
template <typename R>
__global__ __launch_bounds__(kBlock) void k_neq(const typename V2<R>::T *__restrict__ a,
                                                const typename V2<R>::T *__restrict__ b,
                                                uint64_t len, double tol,
                                                double *__restrict__ part) {
  __shared__ double sh[1][kBlock];
  double v[1] = {0.0};
  for (uint64_t i = (uint64_t)blockIdx.x * kBlock + threadIdx.x; i < len;
       i += (uint64_t)gridDim.x * kBlock) {
    const auto x = a[i];
    const auto y = b[i];
    const double dr = (double)x.x - (double)y.x, di = (double)x.y - (double)y.y;
    const double d = hypot(dr, di);
    if (!(d < tol)) v[0] += 1.0;
  }
  block_sum<1>(v, sh);
  if (threadIdx.x == 0) part[blockIdx.x] = v[0];
}

template <typename R>
hipError_t launch_neq_count(const void *a, const void *b, int n, double tol, double *d_part,
                            double *d_out, hipStream_t s) {
  const uint64_t len = 1ull << n;
  const int g = reduce_grid(len);
  hipLaunchKernelGGL(k_neq<R>, dim3(g), dim3(kBlock), 0, s, (const typename V2<R>::T *)a,
                     (const typename V2<R>::T *)b, len, tol, d_part);
  hipLaunchKernelGGL(k_finish<1>, dim3(1), dim3(kBlock), 0, s, (const double *)d_part, g, d_out);
  return hipGetLastError();
}

template <typename R>
__global__ __launch_bounds__(kBlock) void k_probs(const typename V2<R>::T *__restrict__ psi,
                                                  uint64_t len, double *__restrict__ out) {
  for (uint64_t i = (uint64_t)blockIdx.x * kBlock + threadIdx.x; i < len;
       i += (uint64_t)gridDim.x * kBlock) {
    const auto a = psi[i];
    out[i] = (double)a.x * (double)a.x + (double)a.y * (double)a.y;
  }
}

template <typename R>
hipError_t launch_probabilities(const void *psi, int n, double *d_out, hipStream_t s) {
  const uint64_t len = 1ull << n;
  unsigned grid = grid_for(len, kBlock * 4);
  if (grid > 262144) grid = 262144;
  hipLaunchKernelGGL(k_probs<R>, dim3(grid), dim3(kBlock), 0, s, (const typename V2<R>::T *)psi,
                     len, d_out);
  return hipGetLastError();
}

template <typename R>
__global__ __launch_bounds__(kBlock) void k_from_c128(typename V2<R>::T *__restrict__ psi,
                                                      const double *__restrict__ src,
                                                      uint64_t count) {
  for (uint64_t i = (uint64_t)blockIdx.x * kBlock + threadIdx.x; i < count;
       i += (uint64_t)gridDim.x * kBlock) {
    typename V2<R>::T v;
    v.x = (R)src[2 * i];
    v.y = (R)src[2 * i + 1];
    psi[i] = v;
  }
}

template <typename R>
__global__ __launch_bounds__(kBlock) void k_to_c128(double *__restrict__ dst,
                                                    const typename V2<R>::T *__restrict__ psi,
                                                    uint64_t count) {
  for (uint64_t i = (uint64_t)blockIdx.x * kBlock + threadIdx.x; i < count;
       i += (uint64_t)gridDim.x * kBlock) {
    const auto v = psi[i];
    dst[2 * i] = (double)v.x;
    dst[2 * i + 1] = (double)v.y;
  }
}

// Amplitudes at `count` given indices, widened to complex128.
template <typename R>
__global__ __launch_bounds__(kBlock) void k_gather_amps(double *__restrict__ dst,
                                                        const typename V2<R>::T *__restrict__ psi,
                                                        const uint64_t *__restrict__ idx,
                                                        uint64_t count) {
  const uint64_t i = (uint64_t)blockIdx.x * kBlock + threadIdx.x;
  if (i >= count) return;
  const auto v = psi[idx[i]];
  dst[2 * i] = (double)v.x;
  dst[2 * i + 1] = (double)v.y;
}

template <typename R>
hipError_t launch_gather_amps(double *dst, const void *psi, const uint64_t *d_idx, uint64_t count,
                              hipStream_t s) {
  if (count == 0) return hipSuccess;
  hipLaunchKernelGGL(k_gather_amps<R>, dim3(grid_for(count, kBlock)), dim3(kBlock), 0, s, dst,
                     (const typename V2<R>::T *)psi, d_idx, count);
  return hipGetLastError();
}

template <typename R>
hipError_t launch_convert_from_c128(void *psi, const double *src, uint64_t count, hipStream_t s) {
  unsigned grid = grid_for(count, kBlock * 4);
  if (grid > 262144) grid = 262144;
  hipLaunchKernelGGL(k_from_c128<R>, dim3(grid), dim3(kBlock), 0, s, (typename V2<R>::T *)psi, src,
                     count);
  return hipGetLastError();
}

template <typename R>
hipError_t launch_convert_to_c128(double *dst, const void *psi, uint64_t count, hipStream_t s) {
  unsigned grid = grid_for(count, kBlock * 4);
  if (grid > 262144) grid = 262144;
  hipLaunchKernelGGL(k_to_c128<R>, dim3(grid), dim3(kBlock), 0, s, dst,
                     (const typename V2<R>::T *)psi, count);
  return hipGetLastError();
}

// Histogram of |psi|^2 over the bit pattern of m qubits (bin bit j <->
// qubit pos_order[j]).  Block b owns a contiguous range of the free counter
// (the index bits outside the m qubits); thread t owns bins t, t + 256, ...
// and sums them over the block's range in a fixed order, so the result is
// deterministic without atomics.
struct PosList {
  uint8_t p[64];
};

// Histogram of |psi|^2 over the 2^m patterns of the qubits po.p[0..m):
// block b walks the free indices j of its chunk in order; for each j (the
// same for the whole block, so expand() runs on scalar registers) thread t
// loads the amplitudes of its BPT bins (h = t + 256 k) at once, so every
// thread keeps BPT loads in flight.  With fewer than 256 bins, the threads
// of bin h split the chunk S = 256 / 2^m ways (thread t: phase t / 2^m) and
// each phase is a row of its own.  part[(b * S + phase) * 2^m + h].
template <typename R, int BPT>
__global__ __launch_bounds__(kBlock) void k_set_hist(const typename V2<R>::T *__restrict__ psi,
                                                     Fixed fx, PosList po, int m, uint64_t nfree,
                                                     uint64_t per_block,
                                                     double *__restrict__ part) {
  const int H = 1 << m;
  const int S = H >= kBlock ? 1 : kBlock / H;
  const int phase = H >= kBlock ? 0 : (int)threadIdx.x / H;
  // bin h's offset is the deposit of its bits at po.p: the thread's part
  // (bits 0..7 of h, h < 256: one value per thread) ORed with bin k's part
  // (bits 8.. of t + 256 k: the same for every thread, kept on scalar
  // registers), so that a thread holds one 64-bit offset, not BPT
  const int lo_bits = m < 8 ? m : 8;
  const int tl = H >= kBlock ? (int)threadIdx.x : (int)threadIdx.x % H;
  uint64_t dlo = 0;
  for (int b = 0; b < lo_bits; ++b)
    if ((tl >> b) & 1) dlo |= 1ull << po.p[b];
  uint64_t dhi[BPT];
  double acc[BPT];
#pragma unroll
  for (int k = 0; k < BPT; ++k) {
    uint64_t d = 0;
    for (int b = lo_bits; b < m; ++b)
      if (((k * kBlock) >> b) & 1) d |= 1ull << po.p[b];
    dhi[k] = d;
    acc[k] = 0.0;
  }
  const uint64_t j0 = (uint64_t)blockIdx.x * per_block;
  uint64_t j1 = j0 + per_block;
  if (j1 > nfree) j1 = nfree;
  for (uint64_t jj = j0; jj < j1; jj += (uint64_t)S) {
    const uint64_t j = jj + (uint64_t)phase;
    if (j >= j1) break;
    const uint64_t e = expand(j, fx);
    typename V2<R>::T a[BPT];
#pragma unroll
    for (int k = 0; k < BPT; ++k) a[k] = psi[(e | dhi[k]) | dlo];
#pragma unroll
    for (int k = 0; k < BPT; ++k)
      acc[k] += (double)a[k].x * (double)a[k].x + (double)a[k].y * (double)a[k].y;
  }
#pragma unroll
  for (int k = 0; k < BPT; ++k) {
    const int h = H >= kBlock ? (int)threadIdx.x + k * kBlock : (int)threadIdx.x % H;
    part[((size_t)blockIdx.x * S + phase) * H + h] = acc[k];
  }
}

// Column sums of rows x H partials: a workgroup takes bw = min(H, 32) columns
// (256-byte runs) and splits the rows over 256 / bw slices, added in order in
// LDS.  Bound by the read.  1024 rows of 4096: 10 us, 256 with one thread per
// column and 16 workgroups.
__global__ __launch_bounds__(kBlock) void k_hist_finish(const double *__restrict__ part,
                                                        int rows, int H, int bw,
                                                        double *__restrict__ out) {
  __shared__ double sh[kBlock];
  const int c = (int)threadIdx.x % bw, sl = (int)threadIdx.x / bw, ns = kBlock / bw;
  const int h = (int)blockIdx.x * bw + c;
  int r = (int)((long long)rows * sl / ns);
  const int end = (int)((long long)rows * (sl + 1) / ns);
  double v = 0.0;
  for (; r + 7 < end; r += 8) {
    double x[8];
#pragma unroll
    for (int k = 0; k < 8; ++k) x[k] = part[(size_t)(r + k) * H + h];
#pragma unroll
    for (int k = 0; k < 8; ++k) v += x[k];
  }
  for (; r < end; ++r) v += part[(size_t)r * H + h];
  sh[threadIdx.x] = v;
  __syncthreads();
  if (sl == 0) {
    for (int k = 1; k < ns; ++k) v += sh[k * bw + c];
    out[h] = v;
  }
}

// d_part holds blocks * max(1, 256 / 2^m) rows of 2^m partial sums.
template <typename R>
hipError_t launch_set_histogram(const void *psi, int n, const Fixed &fx, const uint8_t *pos_order,
                                int m, double *d_part, int blocks, double *d_hist,
                                hipStream_t s) {
  const int H = 1 << m;
  if (m > 12) return hipErrorInvalidValue;
  const uint64_t nfree = 1ull << (n - m);
  const uint64_t per_block = (nfree + blocks - 1) / blocks;
  PosList po{};
  for (int j = 0; j < m; ++j) po.p[j] = pos_order[j];
  const int bpt = H >= kBlock ? H / kBlock : 1;
  const int rows = blocks * (H >= kBlock ? 1 : kBlock / H);
  using T = typename V2<R>::T;
  auto kern = bpt == 1 ? k_set_hist<R, 1>
              : bpt == 2 ? k_set_hist<R, 2>
              : bpt == 4 ? k_set_hist<R, 4>
              : bpt == 8 ? k_set_hist<R, 8>
                         : k_set_hist<R, 16>;
  hipLaunchKernelGGL(kern, dim3(blocks), dim3(kBlock), 0, s, (const T *)psi, fx, po, m, nfree,
                     per_block, d_part);
  const int bw = std::min(H, 32);
  hipLaunchKernelGGL(k_hist_finish, dim3(H / bw), dim3(kBlock), 0, s, (const double *)d_part, rows,
                     H, bw, d_hist);
  return hipGetLastError();
}

// |psi|^2 of the amplitudes expand(j, fx) for j < count.
template <typename R>
__global__ __launch_bounds__(kBlock) void k_gather_probs(const typename V2<R>::T *__restrict__ psi,
                                                         Fixed fx, uint64_t count,
                                                         double *__restrict__ out) {
  for (uint64_t j = (uint64_t)blockIdx.x * kBlock + threadIdx.x; j < count;
       j += (uint64_t)gridDim.x * kBlock) {
    const auto a = psi[expand(j, fx)];
    out[j] = (double)a.x * (double)a.x + (double)a.y * (double)a.y;
  }
}

template <typename R>
hipError_t launch_gather_probs(const void *psi, const Fixed &fx, uint64_t count, double *d_out,
                               hipStream_t s) {
  unsigned grid = grid_for(count, kBlock);
  if (grid > 65536) grid = 65536;
  hipLaunchKernelGGL(k_gather_probs<R>, dim3(grid), dim3(kBlock), 0, s,
                     (const typename V2<R>::T *)psi, fx, count, d_out);
  return hipGetLastError();
}

template <typename R>
__global__ __launch_bounds__(kBlock) void k_collapse_to(typename V2<R>::T *__restrict__ psi,
                                                        uint64_t len, uint64_t idx, double sq) {
  using T = typename V2<R>::T;
  for (uint64_t i = (uint64_t)blockIdx.x * kBlock + threadIdx.x; i < len;
       i += (uint64_t)gridDim.x * kBlock) {
    if (i == idx) {
      T a = psi[i];
      a.x = (R)((double)a.x / sq);
      a.y = (R)((double)a.y / sq);
      psi[i] = a;
    } else {
      psi[i] = czero<T>();
    }
  }
}

template <typename R>
hipError_t launch_collapse_to(void *psi, int n, uint64_t idx, double total, hipStream_t s) {
  const uint64_t len = 1ull << n;
  unsigned grid = grid_for(len, kBlock * 4);
  if (grid > 262144) grid = 262144;
  hipLaunchKernelGGL(k_collapse_to<R>, dim3(grid), dim3(kBlock), 0, s, (typename V2<R>::T *)psi,
                     len, idx, sqrt(total));
  return hipGetLastError();
}

// One block per chunk; each thread adds its amplitudes (256 apart) in index
// order, then a fixed tree.  Chunks of whole trips keep 16 loads in flight
// per thread, in the same order of additions: a state of few chunks (16 of
// them at 20 qubits) is a chain of load latencies otherwise.
template <typename R>
__global__ __launch_bounds__(kBlock) void k_chunk_sums(const typename V2<R>::T *__restrict__ psi,
                                                       uint64_t len, uint64_t chunk,
                                                       double *__restrict__ out) {
  __shared__ double sh[1][kBlock];
  double v[1] = {0.0};
  const uint64_t start = (uint64_t)blockIdx.x * chunk;
  uint64_t end = start + chunk;
  if (end > len) end = len;
  uint64_t i = start + threadIdx.x;
  for (; i + (uint64_t)(kRedLoads - 1) * kBlock < end; i += kRedTrip) {
    typename V2<R>::T a[kRedLoads];
#pragma unroll
    for (int k = 0; k < kRedLoads; ++k) a[k] = psi[i + (uint64_t)k * kBlock];
#pragma unroll
    for (int k = 0; k < kRedLoads; ++k)
      v[0] += (double)a[k].x * (double)a[k].x + (double)a[k].y * (double)a[k].y;
  }
  for (; i < end; i += kBlock) {
    const auto a = psi[i];
    v[0] += (double)a.x * (double)a.x + (double)a.y * (double)a.y;
  }
  block_sum<1>(v, sh);
  if (threadIdx.x == 0) out[blockIdx.x] = v[0];
}

// Inverse-CDF samples, one wave per shot.  Shot j starts in its chunk of the
// state with the running sum `run` of the chunks before it and takes the
// first amplitude at which the sum of |a|^2, added one by one in index
// order, exceeds tau (the host's scan of the chunk, with the same additions
// in the same order, so the same index).  If rounding leaves the sum at or
// below tau, the chunk's last amplitude with a probability above 0 is taken
// (its last amplitude if there is none).
//
// The chain of dependent FP64 additions bounds a shot (65536 of them for a
// whole chunk), so the shots run side by side, and the next kSampleTrip
// amplitudes load while the current ones are added.  Every lane runs the same
// chain; each row of 16 lanes holds the next 16 values and hands them round
// by DPP.  1000 shots of 26 qubits, complex128: 543 us, 620 with every value
// read from LDS by all lanes (four waves of a CU share its LDS); with the
// readouts beside it 1.39 ms, against 110 ms with the ~640 hit chunks'
// probabilities copied to and scanned on the host.  (A few shots are: see
// sample_on_host.)
constexpr int kSampleLoads = 16;
constexpr int kSampleTrip = 64 * kSampleLoads;
constexpr int kSampleGroup = 64;  // additions between two looks at the sum

// Value of lane K of each row of 16 lanes, on all lanes of the row.
template <int K>
__device__ __forceinline__ double row_bcast(double v) {
  return __builtin_amdgcn_mov_dpp(v, 0x150 + K, 0xF, 0xF, false);  // row_newbcast
}

// sum + v of lane 0 + v of lane 1 + ... of the row, one after the other.
template <int... K>
__device__ __forceinline__ double add_row(double sum, double v, std::integer_sequence<int, K...>) {
  ((sum += row_bcast<K>(v)), ...);
  return sum;
}

template <typename R>
__global__ __launch_bounds__(64) void k_sample(const typename V2<R>::T *__restrict__ psi,
                                               uint64_t chunk, const SampleShot *__restrict__ shots,
                                               uint64_t count, uint64_t *__restrict__ out) {
  using T = typename V2<R>::T;
  __shared__ double p[kSampleTrip];
  if (blockIdx.x >= count) return;
  const SampleShot s = shots[blockIdx.x];
  const T *src = psi + s.chunk * chunk;
  const int lane = threadIdx.x;
  const double tau = s.tau;
  double run = s.run;
  uint64_t last = 0;  // this lane's last index (plus 1) with a probability above 0
  T a[kSampleLoads];
#pragma unroll
  for (int k = 0; k < kSampleLoads; ++k) {
    const uint64_t i = (uint64_t)k * 64 + lane;
    a[k] = i < chunk ? src[i] : czero<T>();
  }
  for (uint64_t w = 0; w < chunk; w += kSampleTrip) {
#pragma unroll
    for (int k = 0; k < kSampleLoads; ++k) {
      const double pr = (double)a[k].x * (double)a[k].x + (double)a[k].y * (double)a[k].y;
      p[k * 64 + lane] = pr;
      if (pr > 0.0) last = w + (uint64_t)k * 64 + lane + 1;
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < kSampleLoads; ++k) {
      const uint64_t i = w + kSampleTrip + (uint64_t)k * 64 + lane;
      a[k] = i < chunk ? src[i] : czero<T>();
    }
    // amplitudes past the chunk's end add 0; they cannot be the first above
    // tau, which an addition of 0 does not reach
    double v[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) v[k] = p[16 * k + (lane & 15)];
    for (int g = 0; g < kSampleTrip; g += kSampleGroup) {
      // the next group's reads are in flight while this one is added (the
      // last group reads itself again)
      double ahead[4];
      const int ag = g + kSampleGroup < kSampleTrip ? g + kSampleGroup : g;
#pragma unroll
      for (int k = 0; k < 4; ++k) ahead[k] = p[ag + 16 * k + (lane & 15)];
      double next = run;
#pragma unroll
      for (int k = 0; k < 4; ++k) next = add_row(next, v[k], std::make_integer_sequence<int, 16>{});
      // not `next > tau`: a NaN behind the first sum above tau must not hide it
      if (!(next <= tau)) {
        double t = run;
        for (int k = 0; k < kSampleGroup; ++k) {
          t += p[g + k];
          if (t > tau) {
            if (lane == 0) out[blockIdx.x] = s.chunk * chunk + w + (uint64_t)(g + k);
            return;  // the same for every lane
          }
        }
      }
      run = next;
#pragma unroll
      for (int k = 0; k < 4; ++k) v[k] = ahead[k];
    }
    __syncthreads();
  }
  for (int d = 32; d > 0; d >>= 1) {
    const uint64_t o = __shfl_xor((unsigned long long)last, d);
    if (o > last) last = o;
  }
  if (lane == 0) out[blockIdx.x] = s.chunk * chunk + (last ? last - 1 : chunk - 1);
}

template <typename R>
hipError_t launch_sample(const void *psi, uint64_t chunk, const SampleShot *d_shots,
                         uint64_t count, uint64_t *d_out, hipStream_t s) {
  if (count == 0) return hipSuccess;
  if (count > 0x7fffffffull) return hipErrorInvalidValue;
  hipLaunchKernelGGL(k_sample<R>, dim3((unsigned)count), dim3(64), 0, s,
                     (const typename V2<R>::T *)psi, chunk, d_shots, count, d_out);
  return hipGetLastError();
}

template <typename R>
hipError_t launch_chunk_sums(const void *psi, int n, uint64_t chunk, double *d_out,
                             hipStream_t s) {
  const uint64_t len = 1ull << n;
  const uint64_t nchunks = (len + chunk - 1) / chunk;
  hipLaunchKernelGGL(k_chunk_sums<R>, dim3((unsigned)nchunks), dim3(kBlock), 0, s,
                     (const typename V2<R>::T *)psi, len, chunk, d_out);
  return hipGetLastError();
}

#define QS_INSTANTIATE(R)                                                                        \
  template hipError_t launch_init_basis<R>(void *, int, uint64_t, hipStream_t);                 \
  template hipError_t launch_init_product<R>(void *, int, const ProductState &, hipStream_t);   \
  template hipError_t launch_zero_outside<R>(void *, int, uint64_t, uint64_t, hipStream_t);     \
  template hipError_t launch_gate_dense<R>(void *, int, const Gate &, void *, void *,            \
                                           hipStream_t);                                         \
  template hipError_t launch_gate_diag<R>(void *, int, const Gate &, void *, hipStream_t);      \
  template hipError_t launch_gate_sparse<R>(void *, int, const Gate &, hipStream_t);            \
  template hipError_t launch_gate_perm<R>(void *, int, const Gate &, const void *, void *,       \
                                          hipStream_t);                                          \
  template hipError_t launch_prob_split<R>(void *, int, int, double *, const SplitEnd &,        \
                                           hipStream_t);                                         \
  template hipError_t launch_collapse<R>(void *, int, int, int, double, hipStream_t);           \
  template hipError_t launch_collapse_pattern<R>(void *, int, uint64_t, uint64_t, double,        \
                                                 hipStream_t);                                   \
  template hipError_t launch_collapse_split<R>(void *, int, int, int, double, int, double *,     \
                                               const SplitEnd &, hipStream_t);                   \
  template hipError_t launch_measure_deferred<R>(void *, int, int, double, double *, double *,  \
                                                 unsigned *, unsigned char *, hipStream_t);     \
  template hipError_t launch_norm<R>(const void *, int, double *, double *, hipStream_t);       \
  template hipError_t launch_neq_count<R>(const void *, const void *, int, double, double *,    \
                                          double *, hipStream_t);                                \
  template hipError_t launch_probabilities<R>(const void *, int, double *, hipStream_t);        \
  template hipError_t launch_convert_from_c128<R>(void *, const double *, uint64_t,             \
                                                  hipStream_t);                                  \
  template hipError_t launch_convert_to_c128<R>(double *, const void *, uint64_t, hipStream_t); \
  template hipError_t launch_gather_amps<R>(double *, const void *, const uint64_t *, uint64_t,  \
                                            hipStream_t);                                       \
  template hipError_t launch_set_histogram<R>(const void *, int, const Fixed &, const uint8_t *, \
                                              int, double *, int, double *, hipStream_t);        \
  template hipError_t launch_gather_probs<R>(const void *, const Fixed &, uint64_t, double *,    \
                                             hipStream_t);                                       \
  template hipError_t launch_collapse_to<R>(void *, int, uint64_t, double, hipStream_t);        \
  template hipError_t launch_sample<R>(const void *, uint64_t, const SampleShot *, uint64_t,     \
                                       uint64_t *, hipStream_t);                                 \
  template hipError_t launch_chunk_sums<R>(const void *, int, uint64_t, double *, hipStream_t);

QS_INSTANTIATE(double)
QS_INSTANTIATE(float)

}  // namespace qs
