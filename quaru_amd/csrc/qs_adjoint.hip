// qs_adjoint.hip -- adjoint-method gradients of <psi(theta)|H|psi(theta)>.
//
// The reference has no differentiation (quaru 0.2.0 only has the OpenQASM U
// gate as a parameterised operation, src/openqasm.rs:145-163, whose
// conventions the rotations here follow: RY(t) = u(t, 0, 0), RZ(t) =
// u(0, 0, t)).
//
// Batch layout: B parameter sets are padded to Bp = 2^nb states stored back
// to back, [Bp][2^n]; the batch index is then nb extra high index bits, so a
// fixed gate on qubit q < n is one launch of the ordinary gate kernels over
// n + nb "qubits".  Rotations carry one matrix per batch element.  The sweeps,
// the reverse blocks and the reductions run over the first B states only: a
// batch of 33 pays for 33 states, not 64 (18 qubits, 4 layers, complex128:
// 2.39 ms a pass, 2.63 with the padding).
//
// Forward:  psi_b = U_N ... U_1 |0>,  E_b = sum_x |psi_b(x)|^2 h(x) with
//           h(x) = sum_t c_t (-1)^popcount(x & mask_t).
// Backward (one reverse sweep, no per-parameter reruns):
//           lambda = h . psi; for i = N..1:
//             rotation i on parameter p:  g_p += Im <lambda| sigma |psi>
//               (= 2 Re <lambda| dU_i/dtheta U_i^dagger |psi>, with
//                dU/dtheta = -(i/2) sigma U),
//             then psi <- U_i^dagger psi, lambda <- U_i^dagger lambda
//           (the three steps are one fused pass over psi and lambda).
// Checkpoints: with checkpoint_every = L > 0 the forward keeps psi after
// every L-th layer, and the backward re-anchors psi to that copy when it
// reaches it, bounding the rounding drift of the uncompute (and, in
// complex64, keeping the reverse sweep within the forward's accuracy).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdlib>
#include <cstring>
#include <vector>

#include "../../include/quaru_hip.h"
#include "qs_internal.h"
#include "qs_sweep.h"
#include "qs_sweep_kernel.h"

namespace {

template <typename R>
struct AV2;
template <>
struct AV2<double> {
  using T = double2;
};
template <>
struct AV2<float> {
  using T = float2;
};

constexpr int kBlock = 256;
constexpr int kItems = 4;

struct POp {
  int kind = 0;  // 0 fixed gate, 1 rotation
  int axis = 0;
  int target = 0;
  size_t param = 0;
  qs::Gate fwd, inv;
  bool unitary = true;  // to 1e-13 (inv undoes fwd)
  int rot_slot = -1;
};

int fail_arg(const char *msg) { return qs::set_error(QS_ERR_ARGUMENT, 0, 0, msg); }

__device__ __forceinline__ uint64_t insert0(uint64_t p, int q) {
  const uint64_t lo = p & ((1ull << q) - 1ull);
  return ((p ^ lo) << 1) | lo;
}

__device__ __forceinline__ uint32_t insert0_32(uint32_t p, uint32_t q) {
  return p + (p & ~((1u << q) - 1u));
}

template <typename R>
__global__ __launch_bounds__(kBlock) void k_init_zero_states(typename AV2<R>::T *psi, int n,
                                                             uint64_t total) {
  for (uint64_t i = (uint64_t)blockIdx.x * kBlock + threadIdx.x; i < total;
       i += (uint64_t)gridDim.x * kBlock) {
    typename AV2<R>::T v;
    v.x = ((i & ((1ull << n) - 1ull)) == 0) ? (R)1 : (R)0;
    v.y = 0;
    psi[i] = v;
  }
}

__global__ __launch_bounds__(kBlock) void k_htable(double *h, int n,
                                                   const unsigned long long *__restrict__ masks,
                                                   const double *__restrict__ coeffs,
                                                   int nterms) {
  const uint64_t len = 1ull << n;
  for (uint64_t x = (uint64_t)blockIdx.x * kBlock + threadIdx.x; x < len;
       x += (uint64_t)gridDim.x * kBlock) {
    double v = 0.0;
    for (int t = 0; t < nterms; ++t)
      v += (__popcll((unsigned long long)x & masks[t]) & 1) ? -coeffs[t] : coeffs[t];
    h[x] = v;
  }
}

// Rotation with one 2x2 matrix per batch element (mats[b*4 + e], complex).
// Work item w is pair p = w mod 2^(n-1) of state b = w >> (n - 1).
template <typename R>
__global__ __launch_bounds__(kBlock) void k_rot(typename AV2<R>::T *__restrict__ psi, int n,
                                                int q, const typename AV2<R>::T *__restrict__ mats,
                                                uint64_t total_pairs) {
  using T = typename AV2<R>::T;
  const uint64_t base = (uint64_t)blockIdx.x * (kBlock * kItems) + threadIdx.x;
  const uint64_t pmask = (1ull << (n - 1)) - 1ull;
#pragma unroll
  for (int it = 0; it < kItems; ++it) {
    const uint64_t w = base + (uint64_t)it * kBlock;
    if (w >= total_pairs) break;
    const uint64_t b = w >> (n - 1), p = w & pmask;
    const uint64_t off = b << n;
    const uint64_t i0 = off | insert0(p, q), i1 = i0 | (1ull << q);
    const T m0 = mats[4 * b], m1 = mats[4 * b + 1], m2 = mats[4 * b + 2], m3 = mats[4 * b + 3];
    const T x = psi[i0], y = psi[i1];
    T u, v;
    u.x = m0.x * x.x - m0.y * x.y + m1.x * y.x - m1.y * y.y;
    u.y = m0.x * x.y + m0.y * x.x + m1.x * y.y + m1.y * y.x;
    v.x = m2.x * x.x - m2.y * x.y + m3.x * y.x - m3.y * y.y;
    v.y = m2.x * x.y + m2.y * x.x + m3.x * y.y + m3.y * y.x;
    psi[i0] = u;
    psi[i1] = v;
  }
}

// One reverse step of a rotation: accumulate Im <lam|sigma|psi> per batch
// element into part[b * nblk + blockIdx.x], then apply U^dagger to psi and
// lam.  grid = (nblk, B); block x covers pairs [x*per, (x+1)*per) of state b.
template <typename R>
__global__ __launch_bounds__(kBlock) void k_rot_reverse(typename AV2<R>::T *__restrict__ psi,
                                                        typename AV2<R>::T *__restrict__ lam,
                                                        int n, int q, int axis,
                                                        const typename AV2<R>::T *__restrict__ mats,
                                                        uint64_t pairs_per_state, uint64_t per,
                                                        double *__restrict__ part) {
  using T = typename AV2<R>::T;
  __shared__ double sh[kBlock];
  const uint64_t b = blockIdx.y;
  const uint64_t off = b << n;
  const T m0 = mats[4 * b], m1 = mats[4 * b + 1], m2 = mats[4 * b + 2], m3 = mats[4 * b + 3];
  // U^dagger = [[conj m0, conj m2], [conj m1, conj m3]]
  double acc = 0.0;
  const uint64_t p0 = (uint64_t)blockIdx.x * per;
  uint64_t p1 = p0 + per;
  if (p1 > pairs_per_state) p1 = pairs_per_state;
  for (uint64_t p = p0 + threadIdx.x; p < p1; p += kBlock) {
    const uint64_t i0 = off | insert0(p, q), i1 = i0 | (1ull << q);
    const T x0 = psi[i0], x1 = psi[i1];
    const T l0 = lam[i0], l1 = lam[i1];
    // s = sigma . psi
    double s0r, s0i, s1r, s1i;
    if (axis == 0) {
      s0r = x1.x; s0i = x1.y; s1r = x0.x; s1i = x0.y;
    } else if (axis == 1) {
      s0r = x1.y; s0i = -(double)x1.x; s1r = -(double)x0.y; s1i = x0.x;
    } else {
      s0r = x0.x; s0i = x0.y; s1r = -(double)x1.x; s1i = -(double)x1.y;
    }
    // Im(conj(l0) s0 + conj(l1) s1)
    acc += (double)l0.x * s0i - (double)l0.y * s0r + (double)l1.x * s1i - (double)l1.y * s1r;
    T y0, y1, k0, k1;
    y0.x = m0.x * x0.x + m0.y * x0.y + m2.x * x1.x + m2.y * x1.y;
    y0.y = m0.x * x0.y - m0.y * x0.x + m2.x * x1.y - m2.y * x1.x;
    y1.x = m1.x * x0.x + m1.y * x0.y + m3.x * x1.x + m3.y * x1.y;
    y1.y = m1.x * x0.y - m1.y * x0.x + m3.x * x1.y - m3.y * x1.x;
    k0.x = m0.x * l0.x + m0.y * l0.y + m2.x * l1.x + m2.y * l1.y;
    k0.y = m0.x * l0.y - m0.y * l0.x + m2.x * l1.y - m2.y * l1.x;
    k1.x = m1.x * l0.x + m1.y * l0.y + m3.x * l1.x + m3.y * l1.y;
    k1.y = m1.x * l0.y - m1.y * l0.x + m3.x * l1.y - m3.y * l1.x;
    psi[i0] = y0;
    psi[i1] = y1;
    lam[i0] = k0;
    lam[i1] = k1;
  }
  sh[threadIdx.x] = acc;
  __syncthreads();
  for (int w = kBlock / 2; w > 0; w >>= 1) {
    if ((int)threadIdx.x < w) sh[threadIdx.x] += sh[threadIdx.x + w];
    __syncthreads();
  }
  if (threadIdx.x == 0) part[b * gridDim.x + blockIdx.x] = sh[0];
}

// grad[b * P + param] += sum_k part[b * nblk + k]   (grid = B blocks)
__global__ __launch_bounds__(kBlock) void k_grad_accum(const double *__restrict__ part, int nblk,
                                                       double *__restrict__ grad, size_t P,
                                                       size_t param) {
  __shared__ double sh[kBlock];
  const int b = blockIdx.x;
  double v = 0.0;
  for (int k = threadIdx.x; k < nblk; k += kBlock) v += part[(size_t)b * nblk + k];
  sh[threadIdx.x] = v;
  __syncthreads();
  for (int w = kBlock / 2; w > 0; w >>= 1) {
    if ((int)threadIdx.x < w) sh[threadIdx.x] += sh[threadIdx.x + w];
    __syncthreads();
  }
  if (threadIdx.x == 0) grad[(size_t)b * P + param] += sh[0];
}

// part[b * nblk + x] = sum over the block's chunk of |psi_b|^2 h
template <typename R>
__global__ __launch_bounds__(kBlock) void k_expect(const typename AV2<R>::T *__restrict__ psi,
                                                   int n, const double *__restrict__ h,
                                                   uint64_t per, double *__restrict__ part) {
  __shared__ double sh[kBlock];
  const uint64_t b = blockIdx.y;
  const uint64_t len = 1ull << n;
  const uint64_t x0 = (uint64_t)blockIdx.x * per;
  uint64_t x1 = x0 + per;
  if (x1 > len) x1 = len;
  double acc = 0.0;
  for (uint64_t x = x0 + threadIdx.x; x < x1; x += kBlock) {
    const auto a = psi[(b << n) | x];
    acc += ((double)a.x * (double)a.x + (double)a.y * (double)a.y) * h[x];
  }
  sh[threadIdx.x] = acc;
  __syncthreads();
  for (int w = kBlock / 2; w > 0; w >>= 1) {
    if ((int)threadIdx.x < w) sh[threadIdx.x] += sh[threadIdx.x + w];
    __syncthreads();
  }
  if (threadIdx.x == 0) part[b * gridDim.x + blockIdx.x] = sh[0];
}

__global__ __launch_bounds__(kBlock) void k_sum_rows(const double *__restrict__ part, int nblk,
                                                     double *__restrict__ out) {
  __shared__ double sh[kBlock];
  const int b = blockIdx.x;
  double v = 0.0;
  for (int k = threadIdx.x; k < nblk; k += kBlock) v += part[(size_t)b * nblk + k];
  sh[threadIdx.x] = v;
  __syncthreads();
  for (int w = kBlock / 2; w > 0; w >>= 1) {
    if ((int)threadIdx.x < w) sh[threadIdx.x] += sh[threadIdx.x + w];
    __syncthreads();
  }
  if (threadIdx.x == 0) out[b] = sh[0];
}

// lam = h . psi
template <typename R>
__global__ __launch_bounds__(kBlock) void k_apply_h(typename AV2<R>::T *__restrict__ lam,
                                                    const typename AV2<R>::T *__restrict__ psi,
                                                    int n, const double *__restrict__ h,
                                                    uint64_t total) {
  const uint64_t mask = (1ull << n) - 1ull;
  for (uint64_t i = (uint64_t)blockIdx.x * kBlock + threadIdx.x; i < total;
       i += (uint64_t)gridDim.x * kBlock) {
    auto a = psi[i];
    const double hv = h[i & mask];
    a.x = (R)((double)a.x * hv);
    a.y = (R)((double)a.y * hv);
    lam[i] = a;
  }
}

__global__ __launch_bounds__(kBlock) void k_fill_zero(double *p, uint64_t count) {
  for (uint64_t i = (uint64_t)blockIdx.x * kBlock + threadIdx.x; i < count;
       i += (uint64_t)gridDim.x * kBlock)
    p[i] = 0.0;
}

// ---- fused reverse pass.  The reverse sweep runs in blocks of operations
// whose pair targets fit one tile of T qubits (the low qubits always among
// them, for contiguous loads), taken out of order where they commute
// (reverse_blocks).  A workgroup loads its tile of psi and of lambda into
// LDS, runs the block's reverse steps there (each rotation: the tile's share
// of Im <lambda|sigma|psi>, then U^dagger on both; each fixed gate: its
// inverse on both) and writes the tile back: one pass over psi and lambda per
// block instead of one per operation.  The records of a block come in passes
// over the tile:
//  * a diagonal pass: any run of phases, diagonals and Z rotations, on tile
//    qubits or not.  All of them multiply psi and lambda by the same factor
//    of modulus 1, so w(x) = Im(conj(lambda_x) psi_x) is the same before and
//    after each, and the gradient of the Z rotation on qubit q is the sum of
//    (-1)^(x_q) w(x): wave_signed gives the sums of all six lane qubits and
//    the total at once.
//  * a pair pass: one X or Y rotation, or two on different tile qubits, on
//    pairs or quads of amplitudes.
//  * a 2x2 pass: the inverse of a (controlled) fixed 2x2.
constexpr int kRevMaxOps = 192;  // records per block
constexpr int kRevMaxRows = 64;  // rotations per block
constexpr int kRevMaxSlots = 32;  // rotations per block summed by RowSums
constexpr int kRevMaxOff = 16;   // Z rotations off the tile per diagonal pass
constexpr int kRevMaxTile = 16;
constexpr int kRevMaxBits = 11;  // tile of at most 2^11 amplitudes
constexpr uint32_t kRevNone = 255;

// One pass.  REV_ROT: k = first | second << 8 tile bit | X flags << 16 (bit
// 16 the first is an X rotation, bit 17 the second) | a second one << 18;
// rows = row | row2 << 8 | slot << 16, the second's slot the next one.
// REV_U1: rows = index of its record.  REV_DIAGS: rows = index of its RevDiag.
enum : uint32_t { REV_ROT = 1, REV_U1 = 2, REV_DIAGS = 3, REV_PHASE = 4, REV_DIAG = 5, REV_RZ = 6 };

struct RevPass {
  uint32_t kind, k, rows, pad;
};

// A diagonal pass: rz[k] = the row of the Z rotation on tile bit k (kRevNone:
// none); lane_row: word offset of 64 bytes, the row that each lane's sum goes
// to (kRevNone: none); the Z rotations off the tile, off[o0 .. o0 + noff) = row |
// qubit << 8; sign: word offset of the tile's sign table, one bit per
// amplitude, the parity of the phases of -1 with patterns on the tile alone
// (~0: none); and records first .. first + count for everything else.
struct RevDiag {
  uint32_t nrz, sign, o0, noff, first, count, lane_row, pad;
  uint32_t rz[kRevMaxTile];
};

// A phase, a diagonal, a further Z rotation on a qubit, or a 2x2.
struct RevRec {
  uint32_t kind;
  uint32_t k;      // tile bit of the target (REV_U1, REV_RZ: kRevNone off the tile)
  uint32_t axis;   // REV_DIAG: number of act bits
  uint32_t out;    // REV_RZ: row of the partial sums
  uint32_t moff;   // values at vals[moff..] as {re, im} pairs
  int32_t a0, a1;  // REV_DIAG: act bits: tile bit (>= 0) or -1 - global qubit; REV_RZ: qubit
  uint32_t slot;   // REV_RZ in complex64
  uint32_t lmask, lval;  // pattern bits on the tile (tile bits)
  uint32_t pad2[2];
  uint64_t umask, uval;  // pattern bits off the tile (global index bits)
};

// The descriptor: header, passes, diagonal passes, records, then values; the
// tables that threads read by their index (row slots, parameters, off-tile Z
// rotations, signs) behind them, at word offset `tab`.
struct RevHeader {
  uint32_t T, npass, nrot, nslot;
  uint32_t ndiag, nrec, tab, params;  // params: word offset of the parameter table
  uint32_t tq[kRevMaxTile];       // tile qubits, ascending
  uint32_t row_of[kRevMaxSlots];  // row of the rotation with that slot
};

// One reverse step of an X or Y rotation on the pair (x0, x1) of psi and
// (l0, l1) of lambda: acc += Im(conj(l0) s0 + conj(l1) s1) with s = sigma .
// psi, then U^dagger on both up to a real factor.  U^dagger is [[c, i s],
// [i s, c]] (X) or [[c, s], [-s, c]] (Y); its entries are divided by the
// larger of c and s in modulus (by s: kSwap), so that each output is one
// multiply-add per component: t = s / c or c / s, |t| <= 1.  The factor is
// the same for the whole tile: it is applied once, when the tile is stored.
// Its errors would be, too, and add up over the blocks: it is 1 / sqrt(1 +
// t^2) for the t that was multiplied by, to twice the precision (factor_rest),
// and so is the product over the tile's rotations.  Root mean square errors of
// gradients against 80-bit arithmetic, 10 layers of 8, 11, 13 qubits: 2.3,
// 2.1, 1.7e-16; 3.5, 3.5, 2.9e-16 with c or s as the factor; 3.1, 3.2, 2.3e-16
// with one kernel per operation.  Backward 1.4% longer than with c or s (20
// qubits, batch 64: 20.65 ms, 20.35).
template <typename R, bool kX, bool kSwap>
__device__ __forceinline__ void rot_reverse_pair(typename AV2<R>::T &x0, typename AV2<R>::T &x1,
                                                 typename AV2<R>::T &l0, typename AV2<R>::T &l1,
                                                 R t, double &acc) {
  using T = typename AV2<R>::T;
  if constexpr (kX)
    acc += (double)l0.x * x1.y - (double)l0.y * x1.x + (double)l1.x * x0.y - (double)l1.y * x0.x;
  else
    acc += (double)l1.x * x0.x + (double)l1.y * x0.y - (double)l0.x * x1.x - (double)l0.y * x1.y;
  auto turn = [t](T &a, T &b) {
    T u, v;
    if constexpr (kX) {
      if constexpr (kSwap) {
        u.x = fma(t, a.x, -b.y);
        u.y = fma(t, a.y, b.x);
        v.x = fma(t, b.x, -a.y);
        v.y = fma(t, b.y, a.x);
      } else {
        u.x = fma(-t, b.y, a.x);
        u.y = fma(t, b.x, a.y);
        v.x = fma(-t, a.y, b.x);
        v.y = fma(t, a.x, b.y);
      }
    } else {
      if constexpr (kSwap) {
        u.x = fma(t, a.x, b.x);
        u.y = fma(t, a.y, b.y);
        v.x = fma(t, b.x, -a.x);
        v.y = fma(t, b.y, -a.y);
      } else {
        u.x = fma(t, b.x, a.x);
        u.y = fma(t, b.y, a.y);
        v.x = fma(-t, a.x, b.x);
        v.y = fma(-t, a.y, b.y);
      }
    }
    a = u;
    b = v;
  };
  turn(x0, x1);
  turn(l0, l1);
}

// The same in complex64: every product and sum rounded as k_rot_reverse
// rounds it (cs = {c, s}, no factor taken out), so that a gradient does not
// depend on how the operations fall into blocks.
template <bool kX>
__device__ __forceinline__ void rot_reverse_pair_f(float2 &x0, float2 &x1, float2 &l0, float2 &l1,
                                                   float2 cs, double &acc) {
  if constexpr (kX)
    acc += (double)l0.x * x1.y - (double)l0.y * x1.x + (double)l1.x * x0.y - (double)l1.y * x0.x;
  else
    acc += (double)l1.x * x0.x + (double)l1.y * x0.y - (double)l0.x * x1.x - (double)l0.y * x1.y;
  const float c = cs.x, s = cs.y;
  auto turn = [c, s](float2 &a, float2 &b) {
    float2 u, v;
    if constexpr (kX) {
      u.x = fmaf(-s, b.y, __fmul_rn(c, a.x));
      u.y = fmaf(s, b.x, __fmul_rn(c, a.y));
      v.x = fmaf(c, b.x, __fmul_rn(-s, a.y));
      v.y = fmaf(c, b.y, __fmul_rn(s, a.x));
    } else {
      u.x = fmaf(s, b.x, __fmul_rn(c, a.x));
      u.y = fmaf(s, b.y, __fmul_rn(c, a.y));
      v.x = fmaf(c, b.x, __fmul_rn(-s, a.x));
      v.y = fmaf(c, b.y, __fmul_rn(-s, a.y));
    }
    a = u;
    b = v;
  };
  turn(x0, x1);
  turn(l0, l1);
}

// U^dagger of a Z rotation on one amplitude, in complex64, rounded as
// k_rot_reverse rounds the bit-clear (s > 0) and the bit-set side.
__device__ __forceinline__ float2 rz_reverse_f(float2 a, float2 cs, bool bit) {
  const float c = cs.x, s = cs.y;
  float2 u;
  if (!bit) {
    u.x = fmaf(c, a.x, __fmul_rn(-s, a.y));
    u.y = fmaf(c, a.y, __fmul_rn(s, a.x));
  } else {
    u.x = fmaf(s, a.y, __fmul_rn(c, a.x));
    u.y = fmaf(-s, a.x, __fmul_rn(c, a.y));
  }
  return u;
}

// The pair step of either precision; cs is the rotation's entry of the
// kernel's table.
template <typename R, bool kX, bool kSwap>
__device__ __forceinline__ void rot_pair(typename AV2<R>::T &x0, typename AV2<R>::T &x1,
                                         typename AV2<R>::T &l0, typename AV2<R>::T &l1,
                                         typename AV2<R>::T cs, double &acc) {
  if constexpr (sizeof(R) == 4)
    rot_reverse_pair_f<kX>(x0, x1, l0, l1, cs, acc);
  else
    rot_reverse_pair<R, kX, kSwap>(x0, x1, l0, l1, cs.x, acc);
}

// Calls f(integral_constant kX, integral_constant kSwap); form bit 0: X, bit
// 1: swapped (the same for the whole wave).
template <typename F>
__device__ __forceinline__ void rot_form(uint32_t form, F &&f) {
  using std::integral_constant;
  if (form & 1u) {
    if (form & 2u)
      f(integral_constant<bool, true>{}, integral_constant<bool, true>{});
    else
      f(integral_constant<bool, true>{}, integral_constant<bool, false>{});
  } else {
    if (form & 2u)
      f(integral_constant<bool, false>{}, integral_constant<bool, true>{});
    else
      f(integral_constant<bool, false>{}, integral_constant<bool, false>{});
  }
}

// The value of one lane, on scalar registers.
__device__ __forceinline__ double read_lane(double v, int lane) {
  const uint64_t b = __double_as_longlong(v);
  const uint32_t lo = __builtin_amdgcn_readlane((uint32_t)b, lane);
  const uint32_t hi = __builtin_amdgcn_readlane((uint32_t)(b >> 32), lane);
  return __longlong_as_double((uint64_t)hi << 32 | lo);
}

// |a + i b|^2 - 1 to twice the precision, for moduli near 1.
__device__ __forceinline__ double norm_error(double a, double b) {
#pragma clang fp contract(off)
  const double p = a * a, q = b * b;
  const double lo = fma(a, a, -p) + fma(b, b, -q);
  return ((p >= q ? (p - 1.0) + q : (q - 1.0) + p)) + lo;
}

// f + lo = 1 / sqrt(1 + t^2) to twice the precision, f being its rounded value
// (with either sign): the factor that makes the pair step's matrix unitary
// for the t that it multiplies by.
__device__ __forceinline__ double factor_rest(double f, double t) {
#pragma clang fp contract(off)
  const double w = f * t, wl = fma(f, t, -w);
  return -0.5 * f * (norm_error(f, w) + 2.0 * w * wl);
}

// A product of such factors, hi + lo.
struct Factor {
  double hi, lo;
};

__device__ __forceinline__ Factor operator*(Factor a, Factor b) {
#pragma clang fp contract(off)
  const double p = a.hi * b.hi;
  const double e = fma(a.lo, b.hi, fma(a.hi, b.lo, fma(a.hi, b.hi, -p)));
  const double hi = p + e;
  return {hi, e - (hi - p)};
}

// Lane l ^ 2^K's value by VALU cross-lane moves.
template <int K>
__device__ __forceinline__ double lane_x(double v) {
  return qs::sweep::lane_xor<K>(v, (threadIdx.x >> K) & 1);
}

// Sums over the lanes for up to 32 rotations of a block, by matrix
// instructions: a 4 x 4 matrix whose row `slot` is ones times a 4 x 4 matrix
// of 16 lanes' values (lanes 16 k + c for k < 4 a column) adds the sums of
// the columns to row `slot` of a 4 x 4 FP64 accumulator; four such products
// side by side take the wave's 64 values.  The 16 columns are added once, at
// the end of the block, so a rotation's share costs one 16-cycle instruction
// instead of a six-step exchange over the wave.
struct RowSums {
  double d[kRevMaxSlots / 4];
};

__device__ __forceinline__ void row_add(RowSums &rs, uint32_t slot, double v) {
  const double a = (threadIdx.x & 3u) == (slot & 3u) ? 1.0 : 0.0;
  const uint32_t g = slot >> 2;  // the same for the whole wave
#pragma unroll
  for (uint32_t i = 0; i < kRevMaxSlots / 4; ++i)
    if (g == i) rs.d[i] = __builtin_amdgcn_mfma_f64_4x4x4f64(a, v, rs.d[i], 0, 0, 0);
}

template <int K>
__device__ __forceinline__ double wht_step(double v) {
  const double o = lane_x<K>(v);
  return ((threadIdx.x >> K) & 1) ? o - v : v + o;
}

// Sums over the wave signed by one lane bit: lane 0 receives the total, lane
// 2^k the sum of (-1)^(bit k of lane) v.  Lane bits 4 and 5 by one matrix
// instruction (rows of ones, of the signs of bit 4 and of bit 5 times the 4 x
// 16 matrix of the lanes' values), bits 0 to 3 by a Walsh-Hadamard butterfly
// over each of those rows.
__device__ __forceinline__ double wave_signed(double v) {
  const uint32_t i = threadIdx.x & 3u, k = (threadIdx.x >> 4) & 3u;
  const double a = i == 3 ? 0.0 : ((i & k) ? -1.0 : 1.0);
  v = __builtin_amdgcn_mfma_f64_4x4x4f64(a, v, 0.0, 0, 0, 0);
  v = wht_step<0>(v);
  v = wht_step<1>(v);
  v = wht_step<2>(v);
  return wht_step<3>(v);
}

// LDS position of tile amplitude j: the low three bits are XORed with the
// next three, so that the strided reads of a pair pass on a low tile bit
// spread over the banks.  Linear over XOR: pos(j ^ b) = pos(j) ^ pos(b).
__device__ __forceinline__ uint32_t rev_pos(uint32_t j) { return j ^ ((j >> 3) & 7u); }

// With `hdiag` lambda is not read but begins as hdiag . psi.
//
// One workgroup per tile (grid = ntiles); dynamic LDS 2 x 2^T amplitudes (at
// least 256); PER = max(1, 2^T / 256).  part[tile * nrot + row] = the tile's
// share of the gradient of the rotation with that row.
//
// Bound by vector and LDS work beside the memory pass.  Backward of the
// 20-qubit, 10-layer, batch-64 ansatz, complex128: 20.7 ms in 15 blocks of
// 1.34-1.39 ms (4 GiB of traffic each, 0.81 ms at the card's copy rate).
// Complex64, in strict order: 31 ms in 25 blocks of 1.20 ms.  Steps there in
// complex128, with 0.44 ms copies at four checkpoints and a kernel for lambda
// still outside: 66 ms (55 blocks of 1.11 ms, operations in strict order, one
// exchange and one descriptor fetch per rotation); 34.5 ms with commuting
// blocks and diagonal passes (2280 instructions per wave); 28.4 ms with
// descriptors fetched ahead, cosines and sines in LDS and sums on the matrix
// cores (by 16 x 16 FP64 products instead of 4 x 4: 35.7 ms); 24.2 ms with one
// multiply-add per component and tables for signs and lane sums (1490
// instructions, the vector units 51% busy).  Tiles of 2^11 complex128
// amplitudes, two workgroups per CU: 27.3 ms then.
template <typename R, int PER>
__global__ __launch_bounds__(kBlock)
__attribute__((amdgpu_waves_per_eu(PER < 8 ? 4 : (sizeof(R) == 8 ? 2 : 3)))) void k_reverse_tile(typename AV2<R>::T *__restrict__ psi,
                                                         typename AV2<R>::T *__restrict__ lam,
                                                         int n, const char *__restrict__ blob_g,
                                                         const typename AV2<R>::T *__restrict__ rot,
                                                         uint64_t Bp, double *__restrict__ part,
                                                         const double *__restrict__ hdiag) {
  using T = typename AV2<R>::T;
  constexpr int PB = PER == 1 ? 0 : (PER == 2 ? 1 : (PER == 4 ? 2 : 3));  // bits of i
  constexpr bool kExact = sizeof(R) == 4;  // complex64: see rot_reverse_pair_f
  extern __shared__ unsigned char rev_smem[];
  __shared__ double rows[kRevMaxRows][kBlock / 64];  // per wave, summed at the end
  // per rotation: X and Y {t, factor} and form (rot_reverse_pair), Z {cos, sin}
  // of half the angle; scale[s]: the square of the factors of the slots below
  __shared__ T cs[kRevMaxRows];
  __shared__ double rest[kRevMaxRows];  // of the factors, below their last bit
  __shared__ uint32_t form[kRevMaxRows];
  __shared__ double scale[kRevMaxSlots + 1];
  // what is the same for every lane is read through the constant address
  // space, on scalar loads
  const QS_CONST char *blob = (const QS_CONST char *)blob_g;
  const QS_CONST RevHeader &h = *(const QS_CONST RevHeader *)blob;
  const QS_CONST RevPass *passes = (const QS_CONST RevPass *)(blob + sizeof(RevHeader));
  const QS_CONST RevDiag *diags = (const QS_CONST RevDiag *)(passes + h.npass);
  const QS_CONST RevRec *recs = (const QS_CONST RevRec *)(diags + h.ndiag);
  const QS_CONST R *vals = (const QS_CONST R *)(recs + h.nrec);
  const uint32_t *tab = (const uint32_t *)blob_g + h.tab;
  const int Tt = (int)h.T;
  const uint32_t E = 1u << Tt;
  const uint32_t tid = threadIdx.x;
  const int lane = tid & 63, wave = tid >> 6;
  constexpr uint32_t EO = (uint32_t)PER * kBlock;  // lambda lies EO amplitudes behind psi
  T *ps = (T *)rev_smem;
  T *ls = ps + EO;
  const uint64_t tile = blockIdx.x;
  uint64_t base = tile;
  for (int i = 0; i < Tt; ++i) base = insert0(base, (int)h.tq[i]);
  const uint64_t b = base >> n;
  // Amplitude j = tid + 256 i of the tile: the thread index gives its low 8
  // tile bits, i the rest (the same for the whole workgroup).  All loads of
  // the tile are issued before the first is waited for.
  const int tb = Tt < 8 ? Tt : 8;
  uint64_t toff = 0;
  for (int i = 0; i < tb; ++i)
    if ((tid >> i) & 1u) toff |= 1ull << h.tq[i];
  // PER amplitudes per thread (2^T / 256, at least 1: a tile of fewer than
  // 256 amplitudes leaves the other threads idle)
  const bool active = tid < E;
  uint64_t ioff[PER];
#pragma unroll
  for (int i = 0; i < PER; ++i) {
    uint64_t o = 0;
#pragma unroll
    for (int k = 0; k < PB; ++k)
      if ((i >> k) & 1) o |= 1ull << h.tq[8 + k];
    ioff[i] = base | toff | o;
  }
  const uint32_t tpos = rev_pos(tid);
  typedef R V __attribute__((ext_vector_type(2)));
  const V *psv = reinterpret_cast<const V *>(psi), *lav = reinterpret_cast<const V *>(lam);
  V *psl = reinterpret_cast<V *>(ps), *lsl = reinterpret_cast<V *>(ls);
  {
    V xv[PER], lv[PER];
    if (active) {
#pragma unroll
      for (int i = 0; i < PER; ++i) {
        xv[i] = psv[ioff[i]];
        if (!hdiag) lv[i] = lav[ioff[i]];
      }
      if (hdiag) {
        // the first block: lambda = h psi (k_apply_h)
#pragma unroll
        for (int i = 0; i < PER; ++i) {
          const double hv = hdiag[ioff[i] & ((1ull << n) - 1ull)];
          lv[i].x = (R)((double)xv[i].x * hv);
          lv[i].y = (R)((double)xv[i].y * hv);
        }
      }
    }
    // a thread per rotation fetches its angle's cosine and sine: m[0] = c (X,
    // Y) or c - i s (Z); m[2] = -i s (X) or s (Y)
    if (tid < h.nrot) {
      const uint32_t a = tab[tid] >> 30;  // axis
      const R *m = (const R *)(rot + ((uint64_t)(tab[tid] & 0x3fffffffu) * Bp + b) * 4);
      const R c = m[0], s = a == 0 ? -m[5] : (a == 1 ? m[4] : -m[1]);
      const bool swap = !kExact && !(fabs(c) >= fabs(s));
      T v;
      v.x = kExact || a == 2 ? c : (swap ? c / s : s / c);
      v.y = kExact || a == 2 || swap ? s : c;
      cs[tid] = v;
      if constexpr (!kExact) rest[tid] = factor_rest(v.y, v.x);
      form[tid] = (a == 0 ? 1u : 0u) | (swap ? 2u : 0u);
    }
    if (active) {
#pragma unroll
      for (int i = 0; i < PER; ++i) {
        psl[tpos + i * kBlock] = xv[i];
        lsl[tpos + i * kBlock] = lv[i];
      }
    }
  }
  __syncthreads();
  // the factor of the whole tile, and the squares by which the sums taken
  // before it is applied are off: the product over the slots, by one wave
  Factor whole = {1.0, 0.0};
  if constexpr (!kExact) {
    if ((uint32_t)lane < h.nslot) {
      const uint32_t row = h.row_of[lane & (kRevMaxSlots - 1)];
      whole = {cs[row].y, rest[row]};
    }
    // inclusive products
#pragma unroll
    for (int d = 1; d < kRevMaxSlots; d <<= 1) {
      const Factor o = {__shfl_up(whole.hi, d), __shfl_up(whole.lo, d)};
      if (lane >= d) whole = whole * o;
    }
    if (wave == 0 && lane < kRevMaxSlots) {
      scale[lane + 1] = fma(whole.hi, whole.hi, 2.0 * whole.hi * whole.lo);
      if (lane == 0) scale[0] = 1.0;
    }
    whole = {read_lane(whole.hi, kRevMaxSlots - 1), read_lane(whole.lo, kRevMaxSlots - 1)};
  }
  RowSums sums = {};
  const uint32_t npass = h.npass;
  RevPass nx = {passes[0].kind, passes[0].k, passes[0].rows, 0};
  for (uint32_t o = 0; o < npass; ++o) {
    const RevPass r = nx;
    // the next pass's record, fetched during this one (behind the last pass
    // lies more of the descriptor)
    nx.kind = passes[o + 1].kind;
    nx.k = passes[o + 1].k;
    nx.rows = passes[o + 1].rows;
    if (r.kind == REV_ROT) {
      const uint32_t k1 = r.k & 255u, k2 = (r.k >> 8) & 255u;
      const uint32_t row1 = r.rows & 255u, slot1 = (r.rows >> 16) & 255u;
      const T c1 = cs[row1];
      const uint32_t f1 = __builtin_amdgcn_readfirstlane(form[row1]);
      double acc = 0.0, acc2 = 0.0;
      if ((r.k >> 18) & 1u) {
        const uint32_t row2 = (r.rows >> 8) & 255u;
        const T c2 = cs[row2];
        const uint32_t f2 = __builtin_amdgcn_readfirstlane(form[row2]);
        const uint32_t b1 = rev_pos(1u << k1), b2 = rev_pos(1u << k2);
        const uint32_t klo = k1 < k2 ? k1 : k2, khi = k1 < k2 ? k2 : k1;
#pragma unroll
        for (int qi = 0; qi < (PER + 3) / 4; ++qi) {
          const uint32_t q = tid + (uint32_t)qi * kBlock;
          if (PER < 4 && q >= E / 4) break;
          const uint32_t j00 = rev_pos(insert0_32(insert0_32(q, klo), khi));
          const uint32_t j01 = j00 ^ b1, j10 = j00 ^ b2, j11 = j01 ^ b2;
          T x00 = ps[j00], x01 = ps[j01], x10 = ps[j10], x11 = ps[j11];
          T l00 = ls[j00], l01 = ls[j01], l10 = ls[j10], l11 = ls[j11];
          rot_form(f1, [&](auto kx, auto ksw) {
            rot_pair<R, decltype(kx)::value, decltype(ksw)::value>(x00, x01, l00, l01, c1, acc);
            rot_pair<R, decltype(kx)::value, decltype(ksw)::value>(x10, x11, l10, l11, c1, acc);
          });
          rot_form(f2, [&](auto kx, auto ksw) {
            rot_pair<R, decltype(kx)::value, decltype(ksw)::value>(x00, x10, l00, l10, c2, acc2);
            rot_pair<R, decltype(kx)::value, decltype(ksw)::value>(x01, x11, l01, l11, c2, acc2);
          });
          ps[j00] = x00;
          ps[j01] = x01;
          ps[j10] = x10;
          ps[j11] = x11;
          ls[j00] = l00;
          ls[j01] = l01;
          ls[j10] = l10;
          ls[j11] = l11;
        }
        // (sums of the second rotation are off by the first one's factor too)
        row_add(sums, slot1, acc);
        row_add(sums, slot1 + 1, acc2);
      } else {
        const uint32_t bk = rev_pos(1u << k1);
#pragma unroll
        for (int pi = 0; pi < (PER + 1) / 2; ++pi) {
          const uint32_t p = tid + (uint32_t)pi * kBlock;
          if (PER < 2 && p >= E / 2) break;
          const uint32_t j0 = rev_pos(insert0_32(p, k1)), j1 = j0 ^ bk;
          T x0 = ps[j0], x1v = ps[j1], l0 = ls[j0], l1 = ls[j1];
          rot_form(f1, [&](auto kx, auto ksw) {
            rot_pair<R, decltype(kx)::value, decltype(ksw)::value>(x0, x1v, l0, l1, c1, acc);
          });
          ps[j0] = x0;
          ps[j1] = x1v;
          ls[j0] = l0;
          ls[j1] = l1;
        }
        row_add(sums, slot1, acc);
      }
    } else if (r.kind == REV_U1) {
      const QS_CONST RevRec &d = recs[r.rows];
      if ((base & d.umask) == d.uval) {  // the same for the whole workgroup
        const QS_CONST R *v = vals + d.moff;  // row-major 2x2 of the inverse gate
        const uint32_t bk = rev_pos(1u << d.k);
#pragma unroll
        for (int pi = 0; pi < (PER + 1) / 2; ++pi) {
          const uint32_t p = tid + (uint32_t)pi * kBlock;
          if (p >= E / 2) break;
          const uint32_t l0 = insert0_32(p, d.k);
          if ((l0 & d.lmask) != d.lval) continue;
          const uint32_t j0 = rev_pos(l0), j1 = j0 ^ bk;
          T z[2][2] = {{ps[j0], ps[j1]}, {ls[j0], ls[j1]}};
          for (int s = 0; s < 2; ++s) {
            const T x0 = z[s][0], x1 = z[s][1];
            T y0, y1;
            y0.x = v[0] * x0.x - v[1] * x0.y + v[2] * x1.x - v[3] * x1.y;
            y0.y = v[0] * x0.y + v[1] * x0.x + v[2] * x1.y + v[3] * x1.x;
            y1.x = v[4] * x0.x - v[5] * x0.y + v[6] * x1.x - v[7] * x1.y;
            y1.y = v[4] * x0.y + v[5] * x0.x + v[6] * x1.y + v[7] * x1.x;
            z[s][0] = y0;
            z[s][1] = y1;
          }
          ps[j0] = z[0][0];
          ps[j1] = z[0][1];
          ls[j0] = z[1][0];
          ls[j1] = z[1][1];
        }
      }
    } else if constexpr (kExact) {
      // a diagonal pass in complex64: the records one by one, on the thread's
      // amplitudes in registers; the phases of -1 (exact, in any order) first
      const QS_CONST RevDiag &g = diags[r.rows];
      T x[PER], l[PER];
#pragma unroll
      for (int i = 0; i < PER; ++i) {
        x[i] = active ? ps[tpos + (uint32_t)i * kBlock] : T{0, 0};
        l[i] = active ? ls[tpos + (uint32_t)i * kBlock] : T{0, 0};
      }
      if (g.sign != ~0u) {
        const uint32_t *st = tab + g.sign + (tid >> 5);
#pragma unroll
        for (int i = 0; i < PER; ++i)
          if (active && ((st[i * (kBlock / 32)] >> (tid & 31u)) & 1u)) {
            x[i].x = -x[i].x;
            x[i].y = -x[i].y;
            l[i].x = -l[i].x;
            l[i].y = -l[i].y;
          }
      }
      const uint32_t e = g.first + g.count;
      for (uint32_t t = g.first; t < e; ++t) {
        const QS_CONST RevRec &d = recs[t];
        if (d.kind == REV_RZ) {
          const T v = cs[d.out];
          const bool tbit =
              d.k == kRevNone ? (bool)((base >> d.a0) & 1ull) : (bool)((tid >> (d.k & 7u)) & 1u);
          double acc = 0.0;
#pragma unroll
          for (int i = 0; i < PER; ++i) {
            const bool bit = d.k >= 8 && d.k != kRevNone ? (bool)((i >> (d.k - 8)) & 1) : tbit;
            const double w = (double)l[i].x * x[i].y - (double)l[i].y * x[i].x;
            acc += bit ? -w : w;
            x[i] = rz_reverse_f(x[i], v, bit);
            l[i] = rz_reverse_f(l[i], v, bit);
          }
          row_add(sums, d.slot, acc);
          continue;
        }
        if ((base & d.umask) != d.uval) continue;  // the same for the whole workgroup
        const bool on = (tid & (d.lmask & 255u)) == (d.lval & 255u);
        const uint32_t im = d.lmask >> 8, iv = d.lval >> 8;
#pragma unroll
        for (int i = 0; i < PER; ++i) {
          if (!on || ((uint32_t)i & im) != iv) continue;
          uint32_t vo = d.moff;
          if (d.kind == REV_DIAG) {
            const uint32_t j = tid + (uint32_t)i * kBlock;
            const uint32_t i0 =
                d.a0 >= 0 ? (j >> d.a0) & 1u : (uint32_t)((base >> (-1 - d.a0)) & 1ull);
            const uint32_t i1 =
                d.axis < 2 ? 0u
                           : (d.a1 >= 0 ? (j >> d.a1) & 1u : (uint32_t)((base >> (-1 - d.a1)) & 1ull));
            vo += 2u * (i0 + 2u * i1);
          }
          const R *vg = (const R *)vals + vo;
          const R vr = vg[0], vi = vg[1];
          T y, k;
          y.x = fmaf(vr, x[i].x, -__fmul_rn(vi, x[i].y));
          y.y = fmaf(vr, x[i].y, __fmul_rn(vi, x[i].x));
          k.x = fmaf(vr, l[i].x, -__fmul_rn(vi, l[i].y));
          k.y = fmaf(vr, l[i].y, __fmul_rn(vi, l[i].x));
          x[i] = y;
          l[i] = k;
        }
      }
      if (active) {
#pragma unroll
        for (int i = 0; i < PER; ++i) {
          ps[tpos + (uint32_t)i * kBlock] = x[i];
          ls[tpos + (uint32_t)i * kBlock] = l[i];
        }
      }
    } else {
      // a diagonal pass: the factor of each of this thread's amplitudes as the
      // thread's part (tr, ti) times that of i (fr, fi)
      const QS_CONST RevDiag &g = diags[r.rows];
      double tr = 1.0, ti = 0.0, fr[PER], fi[PER];
#pragma unroll
      for (int i = 0; i < PER; ++i) {
        fr[i] = 1.0;
        fi[i] = 0.0;
      }
      auto turn = [](double &vr, double &vi, double c, double sv) {
        const double nr = vr * c - vi * sv, ni = vr * sv + vi * c;
        vr = nr;
        vi = ni;
      };
      const bool zsums = g.nrz + g.noff != 0;
      uint32_t lane_row = kRevNone;
      if (zsums) lane_row = reinterpret_cast<const uint8_t *>(tab + g.lane_row)[lane];
      if (g.sign != ~0u) {
        const uint32_t *st = tab + g.sign + (tid >> 5);
#pragma unroll
        for (int i = 0; i < PER; ++i)
          if (active && ((st[i * (kBlock / 32)] >> (tid & 31u)) & 1u)) fr[i] = -1.0;
      }
      const uint32_t noff = g.noff;
      uint32_t orow = 0;
      bool oneg = false;
      if (noff) {
        // Z rotations off the tile: lane l (and l + 16, ...) takes entry l,
        // the product over 16 lanes by exchanges
        double c = 1.0, s = 0.0;
        const uint32_t l = (uint32_t)lane & 15u;
        if (l < noff) {
          const uint32_t en = tab[g.o0 + l];
          orow = en & 255u;
          oneg = (base >> (en >> 8)) & 1ull;
          const T v = cs[orow];
          c = v.x;
          s = oneg ? -(double)v.y : (double)v.y;
        }
        auto mul = [&](double oc, double os) { turn(c, s, oc, os); };
        mul(lane_x<0>(c), lane_x<0>(s));
        mul(lane_x<1>(c), lane_x<1>(s));
        if (noff > 4) {
          mul(lane_x<2>(c), lane_x<2>(s));
          mul(lane_x<3>(c), lane_x<3>(s));
          tr = c;
          ti = s;
        } else {
          // entries 0..3 lie in the first quad of every 16 lanes
          tr = __shfl(c, lane & 48);
          ti = __shfl(s, lane & 48);
        }
      }
      if (g.nrz) {
#pragma unroll
        for (int k = 0; k < 8; ++k) {
          if (g.rz[k] == kRevNone) continue;
          const T v = cs[g.rz[k]];
          turn(tr, ti, v.x, ((tid >> k) & 1u) ? -(double)v.y : (double)v.y);
        }
#pragma unroll
        for (int k = 0; k < PB; ++k) {
          if (g.rz[8 + k] == kRevNone) continue;
          const T v = cs[g.rz[8 + k]];
#pragma unroll
          for (int i = 0; i < PER; ++i)
            turn(fr[i], fi[i], v.x, ((i >> k) & 1) ? -(double)v.y : (double)v.y);
        }
      }
      const uint32_t e = g.first + g.count;
      uint32_t nmore = 0;  // Z rotations among the records
      for (uint32_t t = g.first; t < e; ++t) {
        const QS_CONST RevRec &d = recs[t];
        if (d.kind == REV_RZ) {
          ++nmore;
          const T v = cs[d.out];
          if (d.k >= 8 && d.k != kRevNone) {
#pragma unroll
            for (int i = 0; i < PER; ++i)
              turn(fr[i], fi[i], v.x, ((i >> (d.k - 8)) & 1) ? -(double)v.y : (double)v.y);
          } else {
            const bool bit =
                d.k == kRevNone ? (bool)((base >> d.a0) & 1ull) : (bool)((tid >> d.k) & 1u);
            turn(tr, ti, v.x, bit ? -(double)v.y : (double)v.y);
          }
          continue;
        }
        if ((base & d.umask) != d.uval) continue;  // the same for the whole workgroup
        const bool on = (tid & (d.lmask & 255u)) == (d.lval & 255u);
        const uint32_t im = d.lmask >> 8, iv = d.lval >> 8;
        if (d.kind == REV_PHASE) {
          const double pr = vals[d.moff], pi = vals[d.moff + 1];
          const double vr = on ? pr : 1.0, vi = on ? pi : 0.0;
          if (im == 0) {
            turn(tr, ti, vr, vi);
          } else {
#pragma unroll
            for (int i = 0; i < PER; ++i)
              if (((uint32_t)i & im) == iv) turn(fr[i], fi[i], vr, vi);
          }
        } else {
#pragma unroll
          for (int i = 0; i < PER; ++i) {
            if (((uint32_t)i & im) != iv) continue;
            const uint32_t j = tid + (uint32_t)i * kBlock;
            const uint32_t i0 =
                d.a0 >= 0 ? (j >> d.a0) & 1u : (uint32_t)((base >> (-1 - d.a0)) & 1ull);
            const uint32_t i1 =
                d.axis < 2 ? 0u
                           : (d.a1 >= 0 ? (j >> d.a1) & 1u : (uint32_t)((base >> (-1 - d.a1)) & 1ull));
            const R *vg = (const R *)(vals + d.moff) + 2u * (i0 + 2u * i1);
            const double vr = on ? (double)vg[0] : 1.0, vi = on ? (double)vg[1] : 0.0;
            turn(fr[i], fi[i], vr, vi);
          }
        }
      }
      double w[PER];
#pragma unroll
      for (int i = 0; i < PER; ++i) {
        w[i] = 0.0;
        if (active) {
          const uint32_t j = tpos + (uint32_t)i * kBlock;
          const T x = ps[j], l = ls[j];
          w[i] = (double)l.x * x.y - (double)l.y * x.x;
          turn(fr[i], fi[i], tr, ti);
          if (zsums) {
            // back to modulus 1: the roundings of the product are the same in
            // every tile and would add up
            const double c = -0.5 * fma(fi[i], fi[i], fma(fr[i], fr[i], -1.0));
            fr[i] = fma(fr[i], c, fr[i]);
            fi[i] = fma(fi[i], c, fi[i]);
          }
          const R vr = (R)fr[i], vi = (R)fi[i];
          T y, k;
          y.x = vr * x.x - vi * x.y;
          y.y = vr * x.y + vi * x.x;
          k.x = vr * l.x - vi * l.y;
          k.y = vr * l.y + vi * l.x;
          ps[j] = y;
          ls[j] = k;
        }
      }
      if (zsums || nmore) {
        // total and the sums signed by each bit of i over this thread, then
        // over the wave
        double tot = 0.0, di[PB > 0 ? PB : 1] = {};
#pragma unroll
        for (int i = 0; i < PER; ++i) {
          tot += w[i];
#pragma unroll
          for (int k = 0; k < PB; ++k) di[k] += ((i >> k) & 1) ? -w[i] : w[i];
        }
        tot = wave_signed(tot);
        // the total of di[k] on lane 16 k
        double z = 0.0;
        if constexpr (PB > 0) {
#pragma unroll
          for (int k = 0; k < PB; ++k)
            z = __builtin_amdgcn_mfma_f64_4x4x4f64((tid & 3u) == (uint32_t)k ? 1.0 : 0.0, di[k], z,
                                                   0, 0, 0);
          z += lane_x<0>(z);
          z += lane_x<1>(z);
          z += lane_x<2>(z);
          z += lane_x<3>(z);
        }
        if (lane_row != kRevNone) rows[lane_row][wave] = tot;
        const double t6 = (wave & 1) ? -tot : tot, t7 = (wave & 2) ? -tot : tot;
        if (g.nrz) {
          if (lane == 0) {
            if (g.rz[6] != kRevNone) rows[g.rz[6]][wave] = t6;
            if (g.rz[7] != kRevNone) rows[g.rz[7]][wave] = t7;
          }
#pragma unroll
          for (int k = 0; k < PB; ++k)
            if (lane == 16 * k && g.rz[8 + k] != kRevNone) rows[g.rz[8 + k]][wave] = z;
        }
        if (noff) {
          const double t0 = __shfl(tot, 0);
          if ((uint32_t)lane < noff) rows[orow][wave] = oneg ? -t0 : t0;
        }
        if (nmore) {
          for (uint32_t t = g.first; t < e; ++t) {
            const QS_CONST RevRec &d = recs[t];
            if (d.kind != REV_RZ) continue;
            if (d.k == kRevNone) {
              if (lane == 0) rows[d.out][wave] = ((base >> d.a0) & 1ull) ? -tot : tot;
            } else if (d.k >= 8) {
              if (lane == 16 * (int)(d.k - 8)) rows[d.out][wave] = z;
            } else if (d.k >= 6) {
              if (lane == 0) rows[d.out][wave] = d.k == 6 ? t6 : t7;
            } else if (lane == (1 << d.k)) {
              rows[d.out][wave] = tot;
            }
          }
        }
      }
    }
    __syncthreads();
  }
  // row i of an accumulator is on the lanes 16 i .. 16 i + 15
#pragma unroll
  for (uint32_t g = 0; g < kRevMaxSlots / 4; ++g) {
    if (4 * g >= h.nslot) break;
    double t = sums.d[g];
    t += lane_x<0>(t);
    t += lane_x<1>(t);
    t += lane_x<2>(t);
    t += lane_x<3>(t);
    const uint32_t slot = 4 * g + ((uint32_t)lane >> 4);
    if ((lane & 15) == 0 && slot < h.nslot) rows[h.row_of[slot]][wave] = t;
  }
  __syncthreads();
  if (active) {
    V *pso = reinterpret_cast<V *>(psi), *lao = reinterpret_cast<V *>(lam);
#pragma unroll
    for (int i = 0; i < PER; ++i) {
      V x = psl[tpos + i * kBlock], l = lsl[tpos + i * kBlock];
      if constexpr (!kExact) {
        auto times = [&](R v) { return fma(v, whole.hi, v * whole.lo); };
        x = V{times(x.x), times(x.y)};
        l = V{times(l.x), times(l.y)};
      }
      pso[ioff[i]] = x;
      lao[ioff[i]] = l;
    }
  }
  // one row per thread, the workgroup's rows side by side
  if (tid < h.nrot)
    part[tile * h.nrot + tid] =
        (((rows[tid][0] + rows[tid][1]) + rows[tid][2]) + rows[tid][3]) *
        (kExact ? 1.0 : scale[tab[2 * h.nrot + tid]]);
}

// grad[b * P + params[row]] += sum over the tiles of state b of
// part[tile * nrot + row], in a fixed order.  16 waves share the tiles, a
// lane per row, so the rows of a tile are read side by side; rows with the
// same parameter are added in order by the first of them.  grid = batch.
constexpr int kAccumWaves = 16;

__global__ __launch_bounds__(64 * kAccumWaves) void k_rev_accum(
    const double *__restrict__ part, uint32_t nrot, uint64_t tiles_per_state,
    const uint32_t *__restrict__ params, double *__restrict__ grad, size_t P) {
  __shared__ double sh[kAccumWaves][kRevMaxRows];
  const uint64_t b = blockIdx.x;
  const uint32_t row = threadIdx.x & 63, w = threadIdx.x >> 6;
  double v = 0.0;
  if (row < nrot) {
    const double *pr = part + b * tiles_per_state * nrot + row;
    uint64_t i = w;
    for (; i + 7 * kAccumWaves < tiles_per_state; i += 8 * kAccumWaves) {
      double x[8];
#pragma unroll
      for (int k = 0; k < 8; ++k) x[k] = pr[(i + (uint64_t)k * kAccumWaves) * nrot];
#pragma unroll
      for (int k = 0; k < 8; ++k) v += x[k];
    }
    for (; i < tiles_per_state; i += kAccumWaves) v += pr[i * nrot];
  }
  sh[w][row] = v;
  __syncthreads();
  if (threadIdx.x < nrot) {
    double t = 0.0;
    for (int k = 0; k < kAccumWaves; ++k) t += sh[k][row];
    sh[0][row] = t;
  }
  __syncthreads();
  if (threadIdx.x < nrot) {
    const uint32_t p = params[row];
    bool first = true;
    for (uint32_t r = 0; r < row; ++r) first = first && params[r] != p;
    if (first) {
      double t = 0.0;
      for (uint32_t r = row; r < nrot; ++r)
        if (params[r] == p) t += sh[0][r];
      grad[b * P + p] += t;
    }
  }
}

unsigned grid_of(uint64_t work, uint64_t per, unsigned cap = 262144) {
  uint64_t g = (work + per - 1) / per;
  if (g < 1) g = 1;
  if (g > cap) g = cap;
  return (unsigned)g;
}

}  // namespace

struct qs_pcircuit {
  int n = 0;
  std::vector<POp> ops;
  std::vector<size_t> layer_ends;
  size_t nparams = 0;
  int nrot = 0;
};

struct qs_adjoint {
  qs_pcircuit circ;
  int n = 0, nb = 0;
  size_t B = 0, Bp = 1, P = 0;
  int dtype = QS_C128;
  size_t checkpoint_every = 0;
  qs::Workspace *ws = nullptr;  // owns the stream and the descriptor ring
  hipStream_t stream = nullptr;
  // every buffer below comes from take(), which keeps its size for free_ctx
  struct Buf {
    void *p;
    size_t bytes;
  };
  std::vector<Buf> bufs;
  hipError_t take(void **p, size_t bytes) {
    const hipError_t e = qs::pool_malloc(p, bytes, ws->device);
    if (e == hipSuccess) bufs.push_back({*p, bytes});
    return e;
  }
  void *psi = nullptr, *lam = nullptr;
  std::vector<void *> ckpt;
  std::vector<size_t> ckpt_at;  // checkpoint j holds psi after ops [0, ckpt_at[j])
  double *d_h = nullptr;
  void *d_rot = nullptr;        // [nrot][Bp][4] complex, precision of dtype
  void *d_gmat = nullptr;       // diagonal tables of fixed gates (forward, inverse)
  std::vector<size_t> gmat_off; // per op: offset of fwd table, inv table (bytes)
  double *d_part = nullptr;
  size_t part_count = 0;
  double *d_grad = nullptr;
  double *d_rpart = nullptr;  // partial sums of the tiled reverse blocks
  uint64_t rev_blocks = 0, rev_restores = 0;  // of the last backward
  // descriptor ring of the fused forward pass (device + pinned host)
  char *d_ring = nullptr, *h_ring = nullptr;
  size_t ring_cap = 0, ring_off = 0;
  qs::SweepEngine *engine = nullptr;
  uint64_t sweeps = 0, kernels = 0;
  size_t amp_bytes() const { return dtype == QS_C128 ? 16 : 8; }
  size_t state_bytes() const { return amp_bytes() * (Bp << n); }
  size_t used_bytes() const { return amp_bytes() * (B << n); }  // without the padding states
};

namespace {

void free_ctx(qs_adjoint *c) {
  if (!c) return;
  if (c->stream) (void)hipStreamSynchronize(c->stream);
  for (const auto &b : c->bufs) qs::pool_free(b.p, b.bytes, c->ws->device);
  if (c->engine) qs::sweep_engine_free(c->engine);
  qs::workspace_put(c->ws);
  delete c;
}

// Copy host bytes into the descriptor ring; a slot is reused only after the
// stream has drained.
hipError_t ring_upload(qs_adjoint *c, const void *src, size_t bytes, void **dev) {
  const size_t need = (bytes + 255) & ~(size_t)255;
  if (need > c->ring_cap) return hipErrorInvalidValue;
  if (c->ring_off + need > c->ring_cap) {
    const hipError_t e = hipStreamSynchronize(c->stream);
    if (e != hipSuccess) return e;
    c->ring_off = 0;
  }
  char *h = c->h_ring + c->ring_off;
  char *d = c->d_ring + c->ring_off;
  std::memcpy(h, src, bytes);
  c->ring_off += need;
  *dev = d;
  return hipMemcpyAsync(d, h, bytes, hipMemcpyHostToDevice, c->stream);
}

// Copy host bytes to device memory in stream order, through the ring in
// pieces of at most a quarter of it, so that the host source may go away.
hipError_t upload_to(qs_adjoint *c, const void *src, size_t bytes, void *dev) {
  for (size_t off = 0; off < bytes;) {
    const size_t cnt = std::min(bytes - off, c->ring_cap / 4);
    if (c->ring_off + ((cnt + 255) & ~(size_t)255) > c->ring_cap) {
      const hipError_t e = hipStreamSynchronize(c->stream);
      if (e != hipSuccess) return e;
      c->ring_off = 0;
    }
    char *h = c->h_ring + c->ring_off;
    std::memcpy(h, (const char *)src + off, cnt);
    c->ring_off += (cnt + 255) & ~(size_t)255;
    const hipError_t e =
        hipMemcpyAsync((char *)dev + off, h, cnt, hipMemcpyHostToDevice, c->stream);
    if (e != hipSuccess) return e;
    off += cnt;
  }
  return hipSuccess;
}

// The same into a buffer of the pass's own.
hipError_t upload(qs_adjoint *c, const void *src, size_t bytes, void **dev) {
  const hipError_t e = c->take(dev, bytes);
  return e == hipSuccess ? upload_to(c, src, bytes, *dev) : e;
}

// Whether the forward pass runs through the fused sweep engine
// (QS_ADJOINT_SWEEP, default on) or one kernel per operation.
bool adjoint_sweeps() {
  static const bool on = [] {
    const char *v = std::getenv("QS_ADJOINT_SWEEP");
    return !(v && v[0] == '0');
  }();
  return on;
}

// Apply a classified fixed gate over all Bp states (n + nb index bits).
template <typename R>
hipError_t apply_fixed(qs_adjoint *c, void *buf, const qs::Gate &g, const void *d_table) {
  const int ntot = c->n + c->nb;
  switch (g.kind) {
    case qs::Gate::kIdentity: return hipSuccess;
    case qs::Gate::kSparse: return qs::launch_gate_sparse<R>(buf, ntot, g, c->stream);
    case qs::Gate::kDiag:
      return qs::launch_gate_diag<R>(buf, ntot, g, const_cast<void *>(d_table), c->stream);
    case qs::Gate::kDense:
      return qs::launch_gate_dense<R>(buf, ntot, g, nullptr, nullptr, c->stream);
    case qs::Gate::kPerm:  // rejected when the gate is added
      return hipErrorInvalidValue;
  }
  return hipSuccess;
}

#define AJ(expr)                                          \
  do {                                                    \
    e = (expr);                                           \
    if (e != hipSuccess) return qs::set_hip_error(e, #expr); \
  } while (0)

// The forward pass through the fused sweep engine over n + nb qubits: the
// batch index is nb extra high qubits, each rotation a batched 2x2 whose
// matrix the kernel picks by the tile's batch bits (they are never tile
// qubits), each fixed gate an ordinary gate.  The operations between two
// checkpoints go to the planner as one list; the first sweep after a
// checkpoint leaves it where it is and writes to another buffer.  Gates the planner leaves to per-gate kernels run here.
template <typename R>
int forward_sweeps(qs_adjoint *c, const double *thetas) {
  using T = typename AV2<R>::T;
  const int n = c->n, ntot = c->n + c->nb;
  const size_t Bp = c->Bp, B = c->B, P = c->P;
  hipError_t e = hipSuccess;
  if (!c->engine) c->engine = qs::sweep_engine_new();
  qs::SweepRunner run;
  run.n = ntot;
  run.dtype_c64 = c->dtype == QS_C64;
  run.psi = c->psi;
  run.states = B;
  run.stream = c->stream;
  run.upload = [c](const void *src, size_t bytes, void **dev) {
    return ring_upload(c, src, bytes, dev);
  };
  run.single = [c, n, Bp, B](const qs::Gate &g) -> hipError_t {
    ++c->kernels;
    if (g.bmask) {
      std::vector<T> mats(4 * Bp);
      for (size_t k = 0; k < 4 * Bp; ++k) {
        mats[k].x = (R)g.m[k].re;
        mats[k].y = (R)g.m[k].im;
      }
      void *d = nullptr;
      hipError_t e2 = ring_upload(c, mats.data(), mats.size() * sizeof(T), &d);
      if (e2 != hipSuccess) return e2;
      const uint64_t tp = (1ull << (n - 1)) * B;
      hipLaunchKernelGGL(k_rot<R>, dim3(grid_of(tp, kBlock * kItems, 0xffffffffu)),
                         dim3(kBlock), 0, c->stream, (T *)c->psi, n, g.act[0], (const T *)d, tp);
      return hipGetLastError();
    }
    void *tab = nullptr;
    if (g.kind == qs::Gate::kDiag) {
      std::vector<R> v;
      for (const qs::cd &x : g.m) {
        v.push_back((R)x.re);
        v.push_back((R)x.im);
      }
      hipError_t e2 = ring_upload(c, v.data(), v.size() * sizeof(R), &tab);
      if (e2 != hipSuccess) return e2;
    }
    return apply_fixed<R>(c, c->psi, g, tab);
  };
  // every state of the batch starts as |0...0>
  const uint64_t total = B << n;
  run.fresh = true;
  run.known = (1ull << n) - 1ull;
  run.fill = [c, n, ntot, total, &run]() -> hipError_t {
    if (!run.fresh) return qs::launch_zero_outside<R>(c->psi, ntot, run.known, 0, c->stream);
    hipLaunchKernelGGL(k_init_zero_states<R>, dim3(grid_of(total, kBlock * 4)), dim3(kBlock), 0,
                       c->stream, (T *)c->psi, n, total);
    return hipGetLastError();
  };
  run.copy = [c, &run] {
    return hipMemcpyAsync(c->psi, run.src, c->used_bytes(), hipMemcpyDeviceToDevice, c->stream);
  };
  std::vector<qs::Gate> gates;
  size_t layer = 0;
  auto flush = [&]() -> int {
    hipError_t e2 = hipSuccess;
    if (!gates.empty())
      e2 = qs::sweep_execute(c->engine, run, gates, &c->sweeps, &c->kernels);
    if (e2 == hipSuccess) e2 = qs::sweep_settle(run);
    gates.clear();
    if (e2 != hipSuccess) return qs::set_hip_error(e2, "adjoint forward sweeps");
    return QS_OK;
  };
  for (size_t i = 0; i < c->circ.ops.size(); ++i) {
    const POp &op = c->circ.ops[i];
    if (op.kind == 1) {
      qs::Gate g;
      g.kind = qs::Gate::kDense;
      g.na = 1;
      g.act[0] = op.target;
      g.m.resize(4 * Bp);
      for (size_t b = 0; b < Bp; ++b) {
        const double th = b < B ? thetas[b * P + op.param] : 0.0;
        const double cs = std::cos(th / 2.0), sn = std::sin(th / 2.0);
        qs::cd *m = g.m.data() + 4 * b;
        if (op.axis == QS_AXIS_X) {
          m[0] = {cs, 0};
          m[1] = {0, -sn};
          m[2] = {0, -sn};
          m[3] = {cs, 0};
        } else if (op.axis == QS_AXIS_Y) {
          m[0] = {cs, 0};
          m[1] = {-sn, 0};
          m[2] = {sn, 0};
          m[3] = {cs, 0};
        } else {
          m[0] = {cs, -sn};
          m[1] = {0, 0};
          m[2] = {0, 0};
          m[3] = {cs, sn};
        }
      }
      if (Bp > 1) {
        g.bshift = n;
        g.bmask = (uint32_t)(Bp - 1);
      }
      gates.push_back(std::move(g));
    } else if (op.fwd.kind != qs::Gate::kIdentity) {
      gates.push_back(op.fwd);
    }
    while (layer < c->circ.layer_ends.size() && c->circ.layer_ends[layer] == i + 1) {
      ++layer;
      if (c->checkpoint_every > 0 && layer % c->checkpoint_every == 0 &&
          layer < c->circ.layer_ends.size()) {
        const int rc = flush();
        if (rc != QS_OK) return rc;
        // the checkpoint keeps this buffer; the next sweep reads from it and
        // writes to another (20 qubits, batch 64: 28.2 ms with copies of
        // 0.44 ms each, 26.9 without)
        void *next = nullptr;
        AJ(c->take(&next, c->state_bytes()));
        c->ckpt.push_back(c->psi);
        c->ckpt_at.push_back(i + 1);
        run.src = c->psi;
        run.psi = c->psi = next;
      }
    }
  }
  return flush();
}

template <typename R>
int forward_t(qs_adjoint *c, const double *thetas, const uint64_t *masks, const double *coeffs,
              size_t nterms, double *energies) {
  using T = typename AV2<R>::T;
  const int n = c->n;
  const size_t Bp = c->Bp, B = c->B, P = c->P;
  const uint64_t total = (uint64_t)B << n;
  hipError_t e = hipSuccess;
  AJ(c->take(&c->psi, c->state_bytes()));
  // observable table
  {
    AJ(c->take((void **)&c->d_h, sizeof(double) << n));
    void *d_m = nullptr, *d_c = nullptr;
    const uint64_t none = 0;
    AJ(upload(c, nterms ? masks : &none, sizeof(uint64_t) * std::max<size_t>(nterms, 1), &d_m));
    AJ(upload(c, nterms ? coeffs : (const double *)&none,
              sizeof(double) * std::max<size_t>(nterms, 1), &d_c));
    hipLaunchKernelGGL(k_htable, dim3(grid_of(1ull << n, kBlock * 4)), dim3(kBlock), 0, c->stream,
                       c->d_h, n, (const unsigned long long *)d_m, (const double *)d_c,
                       (int)nterms);
    AJ(hipGetLastError());
  }
  // rotation matrices, one per (rotation, batch element)
  const int nrot = c->circ.nrot;
  std::vector<R> rot((size_t)std::max(nrot, 1) * Bp * 8, (R)0);
  for (const POp &op : c->circ.ops) {
    if (op.kind != 1) continue;
    for (size_t b = 0; b < Bp; ++b) {
      const double th = b < B ? thetas[b * P + op.param] : 0.0;
      const double cs = std::cos(th / 2.0), sn = std::sin(th / 2.0);
      double m[8];
      if (op.axis == QS_AXIS_X) {
        const double v[8] = {cs, 0, 0, -sn, 0, -sn, cs, 0};
        std::memcpy(m, v, sizeof(m));
      } else if (op.axis == QS_AXIS_Y) {
        const double v[8] = {cs, 0, -sn, 0, sn, 0, cs, 0};
        std::memcpy(m, v, sizeof(m));
      } else {
        const double v[8] = {cs, -sn, 0, 0, 0, 0, cs, sn};
        std::memcpy(m, v, sizeof(m));
      }
      R *dst = rot.data() + ((size_t)op.rot_slot * Bp + b) * 8;
      for (int k = 0; k < 8; ++k) dst[k] = (R)m[k];
    }
  }
  AJ(c->take(&c->d_rot, rot.size() * sizeof(R)));
  AJ(upload_to(c, rot.data(), rot.size() * sizeof(R), c->d_rot));
  // diagonal tables of the fixed gates
  {
    std::vector<R> tab;
    c->gmat_off.assign(c->circ.ops.size() * 2, 0);
    for (size_t i = 0; i < c->circ.ops.size(); ++i) {
      const POp &op = c->circ.ops[i];
      if (op.kind != 0) continue;
      const qs::Gate *gs[2] = {&op.fwd, &op.inv};
      for (int s = 0; s < 2; ++s) {
        c->gmat_off[2 * i + s] = tab.size() * sizeof(R);
        if (gs[s]->kind == qs::Gate::kDiag)
          for (const qs::cd &v : gs[s]->m) {
            tab.push_back((R)v.re);
            tab.push_back((R)v.im);
          }
      }
    }
    if (tab.empty()) tab.push_back((R)0);
    AJ(c->take(&c->d_gmat, tab.size() * sizeof(R)));
    AJ(upload_to(c, tab.data(), tab.size() * sizeof(R), c->d_gmat));
  }
  const uint64_t pps = 1ull << (n - 1);
  if (adjoint_sweeps()) {
    const int rc = forward_sweeps<R>(c, thetas);
    if (rc != QS_OK) return rc;
  } else {
    hipLaunchKernelGGL(k_init_zero_states<R>, dim3(grid_of(total, kBlock * 4)), dim3(kBlock), 0,
                       c->stream, (T *)c->psi, n, total);
    AJ(hipGetLastError());
  }
  size_t layer = 0;
  for (size_t i = 0; i < c->circ.ops.size() && !adjoint_sweeps(); ++i) {
    const POp &op = c->circ.ops[i];
    if (op.kind == 1) {
      const T *mats = (const T *)c->d_rot + (size_t)op.rot_slot * Bp * 4;
      const uint64_t tp = pps * B;
      hipLaunchKernelGGL(k_rot<R>, dim3(grid_of(tp, kBlock * kItems, 0xffffffffu)), dim3(kBlock),
                         0, c->stream, (T *)c->psi, n, op.target, mats, tp);
      AJ(hipGetLastError());
    } else {
      AJ(apply_fixed<R>(c, c->psi, op.fwd, (const char *)c->d_gmat + c->gmat_off[2 * i]));
    }
    // checkpoint after every checkpoint_every-th layer (not after the last)
    while (layer < c->circ.layer_ends.size() && c->circ.layer_ends[layer] == i + 1) {
      ++layer;
      if (c->checkpoint_every > 0 && layer % c->checkpoint_every == 0 &&
          layer < c->circ.layer_ends.size()) {
        void *cp = nullptr;
        AJ(c->take(&cp, c->state_bytes()));
        AJ(hipMemcpyAsync(cp, c->psi, c->used_bytes(), hipMemcpyDeviceToDevice, c->stream));
        c->ckpt.push_back(cp);
        c->ckpt_at.push_back(i + 1);
      }
    }
  }
  // energies
  const uint64_t len = 1ull << n;
  const uint64_t per = std::min<uint64_t>(len, 1ull << 14);
  const int nblk = (int)((len + per - 1) / per);
  c->part_count = std::max<size_t>((size_t)nblk, (size_t)((pps + 1023) / 1024)) * B;
  AJ(c->take((void **)&c->d_part, c->part_count * sizeof(double)));
  double *d_e = nullptr;
  AJ(c->take((void **)&d_e, B * sizeof(double)));
  hipLaunchKernelGGL(k_expect<R>, dim3(nblk, (unsigned)B), dim3(kBlock), 0, c->stream,
                     (const T *)c->psi, n, c->d_h, per, c->d_part);
  hipLaunchKernelGGL(k_sum_rows, dim3((unsigned)B), dim3(kBlock), 0, c->stream,
                     (const double *)c->d_part, nblk, d_e);
  AJ(hipGetLastError());
  std::vector<double> eh(B);
  AJ(hipMemcpyAsync(eh.data(), d_e, B * sizeof(double), hipMemcpyDeviceToHost, c->stream));
  AJ(hipStreamSynchronize(c->stream));
  if (energies)
    for (size_t b = 0; b < B; ++b) energies[b] = eh[b];
  return QS_OK;
}

// Whether the reverse pass runs in tiled blocks (QS_ADJOINT_FUSED_REVERSE,
// default on) or one kernel per operation.
bool adjoint_fused_reverse() {
  static const bool on = [] {
    const char *v = std::getenv("QS_ADJOINT_FUSED_REVERSE");
    return !(v && v[0] == '0');
  }();
  return on;
}

// Qubits 0 .. low - 1 are on every tile of the reverse blocks: runs of 128
// bytes.  One qubit more (256-byte runs) measured the same per block (20
// qubits, batch 64) and leaves one less for the
// pair targets.
int reverse_low_bits(int dtype) { return dtype == QS_C128 ? 3 : 4; }

// Tile qubits of the reverse blocks: QS_ADJOINT_TILE, default 10 for
// complex128 and 11 for complex64 (32 KiB of LDS for psi and lambda).
int reverse_tile_bits(int dtype) {
  const char *v = std::getenv("QS_ADJOINT_TILE");
  const int t = v ? std::atoi(v) : (dtype == QS_C128 ? 10 : 11);
  return std::max(1, std::min(t, kRevMaxBits));
}

// An operation of the reverse pass: the qubits its inverse touches off the
// diagonal (x) and on it (z); its pair target (-1: none, diagonal); whether
// it has a tile form, and the records and gradient rows that takes.
struct RevItem {
  size_t op = 0;
  uint64_t x = 0, z = 0;
  int pq = -1;
  bool tile_form = true;
  bool barrier = false;
  int records = 1, rows = 0, slots = 0;  // slots: of RowSums, in complex64 Z rotations too
};

//
// A fixed gate that is not unitary keeps its place among all operations, as
// if it touched every qubit: the gradient before it and after it differ.
// (A program may put one in front of the rotations, to prepare a state; what
// the reverse pass does behind it is of no use then.)
RevItem rev_item(const POp &op, size_t index, int n) {
  RevItem it;
  it.op = index;
  if (op.kind == 1) {
    it.rows = it.slots = 1;
    if (op.axis == QS_AXIS_Z) {
      it.z = 1ull << op.target;
    } else {
      it.x = 1ull << op.target;
      it.pq = op.target;
    }
    return it;
  }
  const qs::Gate &g = op.inv;
  uint64_t act = 0;
  for (int j = 0; j < g.na; ++j) act |= 1ull << g.act[j];
  if (g.kind == qs::Gate::kSparse) {
    it.z = g.smask;
    it.records = (int)g.spat.size();
  } else if (g.kind == qs::Gate::kDiag) {
    it.z = act | g.cmask;
    it.tile_form = g.na >= 1 && g.na <= 2;
  } else if (g.kind == qs::Gate::kDense && g.na == 1) {
    it.x = act;
    it.z = g.cmask;
    it.pq = g.act[0];
  } else {
    it.x = act;
    it.z = g.cmask;
    it.tile_form = false;
  }
  it.barrier = !op.unitary;
  if (it.barrier) it.x = (1ull << n) - 1ull;
  return it;
}

// The reverse sweep in tiled blocks (k_reverse_tile).  Between two checkpoint
// restores the operations are taken in reverse order, and a later one moves
// ahead of earlier ones left for another block where it commutes with each of
// them (on every shared qubit both act diagonally): its gradient Im
// <lambda|sigma|psi> is then the same before and after them.  The tile takes
// the pair targets first come, first served while there is room; diagonal
// operations and controls need no tile qubit.  A gate with no tile form (two
// or more dense target qubits) runs on its own once nothing before it is
// left.  On the layered ansatz a block so reaches into the next layers as far
// as its tile's light cone: 20 qubits, 10 layers, checkpoints every two, 15
// blocks (26 in strict order).  Complex64 keeps the strict order, so that
// every amplitude is rounded as if the operations ran one by one.
template <typename R>
int reverse_blocks(qs_adjoint *c) {
  using T = typename AV2<R>::T;
  hipError_t e = hipSuccess;
  const int n = c->n;
  const size_t Bp = c->Bp, B = c->B, P = c->P;
  const int Tt = std::min(reverse_tile_bits(c->dtype), n);
  // at least one tile qubit is left for a pair target above the low ones
  const int low = Tt == n ? Tt : std::min(Tt - 1, reverse_low_bits(c->dtype));
  const uint64_t tiles_per_state = 1ull << (n - Tt);
  const uint64_t ntiles = tiles_per_state * B;
  // rows of partial sums per block: within 64 MiB
  const int rmax =
      (int)std::max<uint64_t>(1, std::min<uint64_t>(kRevMaxRows, (64ull << 20) / (8 * ntiles)));
  if (!c->d_rpart) AJ(c->take((void **)&c->d_rpart, (uint64_t)rmax * ntiles * sizeof(double)));
  const uint64_t lowset = (1ull << low) - 1ull;
  constexpr bool strict = std::is_same<R, float>::value;
  // Whether an operation may run ahead of those that touch bx off the
  // diagonal and bz on it: complex64 keeps the strict order.
  bool ahead = false;  // something was left behind
  auto free_of = [&](const RevItem &it, uint64_t bx, uint64_t bz) {
    return !(strict && ahead) && !(it.x & (bx | bz)) && !(it.z & bx);
  };
  bool made = false;  // whether lambda = h psi is in memory
  std::vector<RevItem> items;  // left, in reverse order
  std::vector<RevItem> block;
  std::vector<RevPass> passes;
  std::vector<RevDiag> diags;
  std::vector<RevRec> recs;
  std::vector<R> vals;
  std::vector<uint32_t> rows, params, row_scale, offs, lane_rows, signs;
  std::vector<char> blob;
  const int sign_words = std::max(1, 1 << std::max(0, Tt - 5));
  // bit j of in_bit[k]: bit k of j (amplitudes j of the tile)
  std::vector<std::vector<uint32_t>> in_bit((size_t)Tt, std::vector<uint32_t>(sign_words, 0));
  for (int k = 0; k < Tt; ++k)
    for (uint32_t j = 0; j < (1u << Tt); ++j)
      if ((j >> k) & 1u) in_bit[k][j >> 5] |= 1u << (j & 31u);

  // Launch the block's operations on a tile with pair targets S.
  auto launch = [&](uint64_t S) -> int {
    RevHeader hd{};
    hd.T = (uint32_t)Tt;
    uint64_t full = S;
    for (int q = 0; q < n && __builtin_popcountll(full) < Tt; ++q) full |= 1ull << q;
    int loc[64];
    int t = 0;
    for (int q = 0; q < 64; ++q) {
      loc[q] = -1;
      if ((full >> q) & 1ull) {
        hd.tq[t] = (uint32_t)q;
        loc[q] = t++;
      }
    }
    passes.clear();
    diags.clear();
    recs.clear();
    vals.clear();
    rows.clear();
    params.clear();
    row_scale.clear();
    offs.clear();
    lane_rows.clear();
    signs.clear();
    auto put = [&](const qs::cd &v) {
      vals.push_back((R)v.re);
      vals.push_back((R)v.im);
    };
    auto pattern = [&](RevRec &r, uint64_t mask, uint64_t val) {
      r.umask = mask & ~full;
      r.uval = val & r.umask;
      for (uint64_t bits = mask & full; bits; bits &= bits - 1) {
        const int q = __builtin_ctzll(bits);
        r.lmask |= 1u << loc[q];
        if ((val >> q) & 1ull) r.lval |= 1u << loc[q];
      }
    };
    auto new_row = [&](const POp &op) {
      rows.push_back((uint32_t)op.rot_slot | ((uint32_t)op.axis << 30));
      params.push_back((uint32_t)op.param);
      row_scale.push_back(hd.nslot);  // the slots before it
      return (uint32_t)rows.size() - 1;
    };
    // a diagonal operation, into the diagonal pass d (signs: its sign table)
    auto emit_diag = [&](const RevItem &it, RevDiag &d, std::vector<uint32_t> &sg) {
      const POp &op = c->circ.ops[it.op];
      const qs::Gate &g = op.inv;
      RevRec r{};
      if (op.kind == 1) {
        r.out = new_row(op);
        const int k = loc[op.target];
        if (strict) {
          r.kind = REV_RZ;
          r.k = k >= 0 ? (uint32_t)k : kRevNone;
          r.a0 = op.target;
          r.slot = hd.nslot++;
          hd.row_of[r.slot] = r.out;
          recs.push_back(r);
        } else if (k >= 0 && d.rz[k] == kRevNone) {
          d.rz[k] = r.out;
          ++d.nrz;
        } else if (k < 0 && d.noff < (uint32_t)kRevMaxOff) {
          offs.push_back(r.out | ((uint32_t)op.target << 8));
          ++d.noff;
        } else {
          r.kind = REV_RZ;
          r.k = k >= 0 ? (uint32_t)k : kRevNone;
          r.a0 = op.target;
          recs.push_back(r);
        }
      } else if (g.kind == qs::Gate::kSparse) {
        for (size_t k = 0; k < g.spat.size(); ++k) {
          if (g.m[k].re == -1.0 && g.m[k].im == 0.0 && (g.smask & ~full) == 0) {
            if (sg.empty()) sg.assign((size_t)sign_words, 0);
            for (int w = 0; w < sign_words; ++w) {
              uint32_t on = ~0u;
              for (uint64_t bits = g.smask; bits; bits &= bits - 1) {
                const int q = __builtin_ctzll(bits);
                const uint32_t m = in_bit[loc[q]][w];
                on &= ((g.spat[k] >> q) & 1ull) ? m : ~m;
              }
              sg[w] ^= on;
            }
            continue;
          }
          RevRec x = r;
          x.kind = REV_PHASE;
          x.moff = (uint32_t)vals.size();
          put(g.m[k]);
          pattern(x, g.smask, g.spat[k]);
          recs.push_back(x);
        }
      } else {
        r.kind = REV_DIAG;
        r.axis = (uint32_t)g.na;
        r.moff = (uint32_t)vals.size();
        for (const qs::cd &v : g.m) put(v);
        pattern(r, g.cmask, g.cval);
        r.a0 = loc[g.act[0]] >= 0 ? loc[g.act[0]] : -1 - g.act[0];
        r.a1 = g.na < 2 ? 0 : (loc[g.act[1]] >= 0 ? loc[g.act[1]] : -1 - g.act[1]);
        recs.push_back(r);
      }
    };
    // passes: by turns every diagonal operation that may come next, and every
    // X / Y rotation that may (two on different qubits to a pass)
    while (!block.empty()) {
      std::vector<RevItem> left;
      std::vector<uint32_t> sg;
      uint64_t bx = 0, bz = 0;
      ahead = false;
      RevDiag d{};
      d.o0 = (uint32_t)offs.size();
      d.first = (uint32_t)recs.size();
      for (uint32_t &v : d.rz) v = kRevNone;
      bool any = false;
      for (const RevItem &it : block) {
        const bool movable = free_of(it, bx, bz);
        if (movable && it.pq < 0 && !(it.barrier && any)) {
          emit_diag(it, d, sg);
          any = true;
          if (it.barrier) bx = it.x;  // alone in its pass
        } else {
          bx |= it.x;
          bz |= it.z;
          left.push_back(it);
          ahead = true;
        }
      }
      if (any) {
        d.count = (uint32_t)recs.size() - d.first;
        d.lane_row = (uint32_t)lane_rows.size();
        uint8_t lr[64];
        std::memset(lr, kRevNone, sizeof lr);
        for (int k = 0; k < std::min(Tt, 6); ++k) lr[1 << k] = (uint8_t)d.rz[k];
        lane_rows.resize(lane_rows.size() + 16);
        std::memcpy(&lane_rows[d.lane_row], lr, sizeof lr);
        d.sign = sg.empty() ? ~0u : (uint32_t)signs.size();
        signs.insert(signs.end(), sg.begin(), sg.end());
        passes.push_back({REV_DIAGS, 0, (uint32_t)diags.size(), 0});
        diags.push_back(d);
      }
      block.swap(left);
      left.clear();
      bx = bz = 0;
      ahead = false;
      size_t open = ~(size_t)0;  // a rotation pass with room for a second
      for (const RevItem &it : block) {
        const bool movable = free_of(it, bx, bz);
        if (!(movable && it.pq >= 0)) {
          bx |= it.x;
          bz |= it.z;
          left.push_back(it);
          ahead = true;
          continue;
        }
        const POp &op = c->circ.ops[it.op];
        const uint32_t k = (uint32_t)loc[it.pq];
        if (op.kind == 1) {
          const uint32_t row = new_row(op), slot = hd.nslot++;
          hd.row_of[slot] = row;
          const uint32_t is_x = op.axis == QS_AXIS_X;
          if (open != ~(size_t)0 && (passes[open].k & 255u) != k) {
            // slots are given in the order of the passes: the second's is the
            // next after the first's
            passes[open].k |= (k << 8) | (is_x << 17) | (1u << 18);
            passes[open].rows |= row << 8;
            open = ~(size_t)0;
          } else {
            open = passes.size();
            passes.push_back({REV_ROT, k | (is_x << 16), row | (slot << 16), 0});
          }
        } else {
          RevRec r{};
          r.kind = REV_U1;
          r.moff = (uint32_t)vals.size();
          for (const qs::cd &v : op.inv.m) put(v);
          pattern(r, op.inv.cmask, op.inv.cval);
          r.k = k;
          passes.push_back({REV_U1, 0, (uint32_t)recs.size(), 0});
          recs.push_back(r);
          open = ~(size_t)0;
        }
      }
      block.swap(left);
    }
    hd.npass = (uint32_t)passes.size();
    hd.nrot = (uint32_t)rows.size();
    hd.ndiag = (uint32_t)diags.size();
    hd.nrec = (uint32_t)recs.size();
    const size_t fixed = sizeof(RevHeader) + passes.size() * sizeof(RevPass) +
                         diags.size() * sizeof(RevDiag) + recs.size() * sizeof(RevRec) +
                         vals.size() * sizeof(R);
    hd.tab = (uint32_t)((fixed + 15) / 16 * 4);
    hd.params = hd.tab + hd.nrot;
    const uint32_t off_at = 3 * hd.nrot, lane_at = off_at + (uint32_t)offs.size(),
                   sign_at = lane_at + (uint32_t)lane_rows.size();
    for (RevDiag &d : diags) {  // offsets from `tab`
      d.o0 += off_at;
      d.lane_row += lane_at;
      if (d.sign != ~0u) d.sign += sign_at;
    }
    blob.assign((size_t)(hd.tab + sign_at) * 4 + signs.size() * 4, 0);
    char *w = blob.data();
    auto add = [&](const void *p, size_t bytes) {
      if (bytes) std::memcpy(w, p, bytes);
      w += bytes;
    };
    add(&hd, sizeof hd);
    add(passes.data(), passes.size() * sizeof(RevPass));
    add(diags.data(), diags.size() * sizeof(RevDiag));
    add(recs.data(), recs.size() * sizeof(RevRec));
    add(vals.data(), vals.size() * sizeof(R));
    w = blob.data() + (size_t)hd.tab * 4;
    add(rows.data(), rows.size() * 4);
    add(params.data(), params.size() * 4);
    add(row_scale.data(), row_scale.size() * 4);
    add(offs.data(), offs.size() * 4);
    add(lane_rows.data(), lane_rows.size() * 4);
    add(signs.data(), signs.size() * 4);
    void *d_blob = nullptr;
    AJ(ring_upload(c, blob.data(), blob.size(), &d_blob));
    const size_t lds = 2 * std::max<size_t>((size_t)1 << Tt, kBlock) * sizeof(T);
    auto kern = Tt <= 8 ? k_reverse_tile<R, 1>
                        : (Tt == 9 ? k_reverse_tile<R, 2>
                                   : (Tt == 10 ? k_reverse_tile<R, 4> : k_reverse_tile<R, 8>));
    hipLaunchKernelGGL(kern, dim3((unsigned)ntiles), dim3(kBlock), lds, c->stream, (T *)c->psi,
                       (T *)c->lam, n, (const char *)d_blob, (const T *)c->d_rot, (uint64_t)Bp,
                       c->d_rpart, made ? nullptr : c->d_h);
    AJ(hipGetLastError());
    made = true;
    ++c->rev_blocks;
    if (!params.empty()) {
      hipLaunchKernelGGL(k_rev_accum, dim3((unsigned)B), dim3(64 * kAccumWaves), 0, c->stream,
                         (const double *)c->d_rpart, (uint32_t)params.size(), tiles_per_state,
                         (const uint32_t *)d_blob + hd.params, c->d_grad, P);
      AJ(hipGetLastError());
    }
    return QS_OK;
  };

  // lambda = h psi for what is not the first block
  auto make = [&]() -> int {
    if (made) return QS_OK;
    made = true;
    const uint64_t total = (uint64_t)B << n;
    hipLaunchKernelGGL(k_apply_h<R>, dim3(grid_of(total, kBlock * 4)), dim3(kBlock), 0, c->stream,
                       (T *)c->lam, (const T *)c->psi, n, c->d_h, total);
    AJ(hipGetLastError());
    return QS_OK;
  };

  // Run everything in `items` (the operations since the last restore).
  auto drain = [&]() -> int {
    std::vector<RevItem> left;
    while (!items.empty()) {
      if (!items[0].tile_form) {
        const size_t ii = items[0].op;
        const qs::Gate &g = c->circ.ops[ii].inv;
        const void *tab = (const char *)c->d_gmat + c->gmat_off[2 * ii + 1];
        const int rc = make();
        if (rc != QS_OK) return rc;
        AJ(apply_fixed<R>(c, c->psi, g, tab));
        AJ(apply_fixed<R>(c, c->lam, g, tab));
        items.erase(items.begin());
        continue;
      }
      block.clear();
      left.clear();
      uint64_t S = lowset, bx = 0, bz = 0;
      ahead = false;
      int nrec = 0, nrow = 0, nslot = 0;
      for (size_t i = 0; i < items.size(); ++i) {
        const RevItem &it = items[i];
        const uint64_t bq = it.pq >= 0 ? 1ull << it.pq : 0;
        const bool movable = free_of(it, bx, bz);
        if (it.tile_form && movable && nrec + it.records <= kRevMaxOps &&
            nrow + it.rows <= rmax && nslot + (strict || it.pq >= 0 ? it.slots : 0) <= kRevMaxSlots &&
            __builtin_popcountll(S | bq) <= Tt) {
          S |= bq;
          nrec += it.records;
          nrow += it.rows;
          nslot += strict || it.pq >= 0 ? it.slots : 0;
          block.push_back(it);
        } else {
          bx |= it.x;
          bz |= it.z;
          if (!it.tile_form) bx |= it.z;
          left.push_back(it);
          ahead = true;
        }
      }
      items.swap(left);
      const int rc = launch(S);
      if (rc != QS_OK) return rc;
    }
    return QS_OK;
  };

  int ck = (int)c->ckpt.size() - 1;
  for (size_t ii = c->circ.ops.size(); ii-- > 0;) {
    if (ck >= 0 && c->ckpt_at[ck] == ii + 1) {
      int rc = drain();
      if (rc == QS_OK) rc = make();
      if (rc != QS_OK) return rc;
      std::swap(c->psi, c->ckpt[ck]);  // the uncomputed state is not needed any more
      ++c->rev_restores;
      --ck;
    }
    const POp &op = c->circ.ops[ii];
    if (op.kind == 0 && op.inv.kind == qs::Gate::kIdentity) continue;
    items.push_back(rev_item(op, ii, n));
  }
  return drain();
}

template <typename R>
int backward_t(qs_adjoint *c, double *grads) {
  using T = typename AV2<R>::T;
  const int n = c->n;
  const size_t Bp = c->Bp, B = c->B, P = c->P;
  const uint64_t total = (uint64_t)B << n;
  hipError_t e = hipSuccess;
  if (!c->lam) AJ(c->take(&c->lam, c->state_bytes()));
  if (!c->d_grad) AJ(c->take((void **)&c->d_grad, B * std::max<size_t>(P, 1) * sizeof(double)));
  hipLaunchKernelGGL(k_fill_zero, dim3(grid_of(B * P, kBlock)), dim3(kBlock), 0, c->stream,
                     c->d_grad, (uint64_t)(B * P));
  AJ(hipGetLastError());
  if (!adjoint_fused_reverse()) {  // the tiled blocks make lambda themselves
    hipLaunchKernelGGL(k_apply_h<R>, dim3(grid_of(total, kBlock * 4)), dim3(kBlock), 0, c->stream,
                       (T *)c->lam, (const T *)c->psi, n, c->d_h, total);
    AJ(hipGetLastError());
  }
  const uint64_t pps = 1ull << (n - 1);
  const uint64_t per = std::min<uint64_t>(pps, 1024);
  const int nblk = (int)((pps + per - 1) / per);
  int ck = (int)c->ckpt.size() - 1;
  c->rev_blocks = c->rev_restores = 0;
  if (adjoint_fused_reverse()) {
    const int rc = reverse_blocks<R>(c);
    if (rc != QS_OK) return rc;
  }
  for (size_t ii = adjoint_fused_reverse() ? 0 : c->circ.ops.size(); ii-- > 0;) {
    if (ck >= 0 && c->ckpt_at[ck] == ii + 1) {
      std::swap(c->psi, c->ckpt[ck]);
      --ck;
    }
    const POp &op = c->circ.ops[ii];
    if (op.kind == 1) {
      const T *mats = (const T *)c->d_rot + (size_t)op.rot_slot * Bp * 4;
      hipLaunchKernelGGL(k_rot_reverse<R>, dim3(nblk, (unsigned)B), dim3(kBlock), 0, c->stream,
                         (T *)c->psi, (T *)c->lam, n, op.target, op.axis, mats, pps, per,
                         c->d_part);
      hipLaunchKernelGGL(k_grad_accum, dim3((unsigned)B), dim3(kBlock), 0, c->stream,
                         (const double *)c->d_part, nblk, c->d_grad, P, op.param);
      AJ(hipGetLastError());
    } else {
      const void *tab = (const char *)c->d_gmat + c->gmat_off[2 * ii + 1];
      AJ(apply_fixed<R>(c, c->psi, op.inv, tab));
      AJ(apply_fixed<R>(c, c->lam, op.inv, tab));
    }
  }
  std::vector<double> g(B * P);
  AJ(hipMemcpyAsync(g.data(), c->d_grad, g.size() * sizeof(double), hipMemcpyDeviceToHost,
                    c->stream));
  AJ(hipStreamSynchronize(c->stream));
  std::memcpy(grads, g.data(), c->B * P * sizeof(double));
  return QS_OK;
#undef AJ
}

}  // namespace

extern "C" {

int qs_pcircuit_new(size_t n, qs_pcircuit **out) {
  if (!out) return fail_arg("out is NULL");
  if (n < 1 || n > 30) return qs::set_error(QS_ERR_ARGUMENT, n, 0, "pcircuit needs 1..30 qubits");
  qs_pcircuit *c = new qs_pcircuit();
  c->n = (int)n;
  *out = c;
  return QS_OK;
}

void qs_pcircuit_free(qs_pcircuit *c) { delete c; }

int qs_pcircuit_gate(qs_pcircuit *c, const double *matrix, const size_t *targets, size_t k) {
  if (!c || !matrix || !targets) return fail_arg("NULL argument");
  if (k < 1 || k > 2) return qs::set_error(QS_INVALID_DIMENSIONS, k, k, "fixed gates: k = 1 or 2");
  std::vector<size_t> t(targets, targets + k);
  if (k == 2 && t[0] == t[1]) return qs::set_error(QS_INVALID_TARGET, t[0], 0, "duplicate target");
  for (size_t j = 0; j < k; ++j)
    if (t[j] >= (size_t)c->n) return qs::set_error(QS_INVALID_TARGET, t[j], 0, "target out of range");
  const size_t D = (size_t)1 << k;
  std::vector<double> inv(2 * D * D);
  for (size_t i = 0; i < D; ++i)
    for (size_t j = 0; j < D; ++j) {
      inv[2 * (i * D + j)] = matrix[2 * (j * D + i)];
      inv[2 * (i * D + j) + 1] = -matrix[2 * (j * D + i) + 1];
    }
  POp op;
  op.kind = 0;
  for (size_t i = 0; i < D; ++i)
    for (size_t j = 0; j < D; ++j) {
      double re = i == j ? -1.0 : 0.0, im = 0.0;  // of row i times row j's conjugate
      for (size_t e = 0; e < D; ++e) {
        const double *a = matrix + 2 * (i * D + e), *b = matrix + 2 * (j * D + e);
        re += a[0] * b[0] + a[1] * b[1];
        im += a[1] * b[0] - a[0] * b[1];
      }
      op.unitary = op.unitary && std::fabs(re) < 1e-13 && std::fabs(im) < 1e-13;
    }
  op.fwd = qs::classify_matrix(matrix, t.data(), k, 0, 0);
  op.inv = qs::classify_matrix(inv.data(), t.data(), k, 0, 0);
  if ((op.fwd.kind == qs::Gate::kDense && op.fwd.na > 2) ||
      (op.fwd.kind == qs::Gate::kDiag && op.fwd.na > 2) || op.fwd.kind == qs::Gate::kPerm)
    return qs::set_error(QS_INVALID_DIMENSIONS, k, k, "unsupported fixed gate");
  c->ops.push_back(std::move(op));
  return QS_OK;
}

int qs_pcircuit_rotation(qs_pcircuit *c, int axis, size_t target, size_t param) {
  if (!c) return fail_arg("NULL argument");
  if (axis < QS_AXIS_X || axis > QS_AXIS_Z) return fail_arg("axis must be 0 (X), 1 (Y) or 2 (Z)");
  if (target >= (size_t)c->n) return qs::set_error(QS_INVALID_TARGET, target, 0, "target out of range");
  POp op;
  op.kind = 1;
  op.axis = axis;
  op.target = (int)target;
  op.param = param;
  op.rot_slot = c->nrot++;
  c->nparams = std::max(c->nparams, param + 1);
  c->ops.push_back(std::move(op));
  return QS_OK;
}

int qs_pcircuit_layer(qs_pcircuit *c) {
  if (!c) return fail_arg("NULL argument");
  c->layer_ends.push_back(c->ops.size());
  return QS_OK;
}

size_t qs_pcircuit_nparams(const qs_pcircuit *c) { return c ? c->nparams : 0; }

int qs_adjoint_forward(const qs_pcircuit *c, const double *thetas, size_t batch,
                       const uint64_t *masks, const double *coeffs, size_t nterms, int dtype,
                       size_t checkpoint_every, qs_adjoint **ctx, double *energies) {
  if (ctx) *ctx = nullptr;
  if (!c || batch == 0 || (c->nparams > 0 && !thetas) || (nterms > 0 && (!masks || !coeffs)))
    return fail_arg("NULL argument or empty batch");
  if (dtype != QS_C128 && dtype != QS_C64) return fail_arg("bad dtype");
  int count = 0;
  if (hipGetDeviceCount(&count) != hipSuccess || count == 0)
    return qs::set_error(QS_ERR_NO_DEVICE, 0, 0, "no HIP device available");
  qs_adjoint *a = new qs_adjoint();
  a->circ = *c;
  a->n = c->n;
  a->B = batch;
  a->Bp = 1;
  a->nb = 0;
  while (a->Bp < batch) {
    a->Bp <<= 1;
    ++a->nb;
  }
  if (a->n + a->nb > qs::kMaxQubits) {
    delete a;
    return fail_arg("batch x state too large");
  }
  a->P = c->nparams;
  a->dtype = dtype;
  a->checkpoint_every = checkpoint_every;
  int device = 0;
  hipError_t e = hipGetDevice(&device);
  if (e == hipSuccess) e = qs::workspace_get(&a->ws, device);
  if (e != hipSuccess) {
    delete a;
    return qs::set_hip_error(e, "adjoint workspace");
  }
  a->stream = a->ws->stream;
  a->d_ring = a->ws->d_ring;
  a->h_ring = a->ws->h_ring;
  a->ring_cap = qs::kRingBytes;
  const int rc = dtype == QS_C128 ? forward_t<double>(a, thetas, masks, coeffs, nterms, energies)
                                  : forward_t<float>(a, thetas, masks, coeffs, nterms, energies);
  if (rc != QS_OK || !ctx) {
    free_ctx(a);
    return rc;
  }
  *ctx = a;
  return QS_OK;
}

int qs_adjoint_backward(qs_adjoint *ctx, double *grads) {
  if (!ctx || !grads) return fail_arg("NULL argument");
  if (ctx->P == 0) return QS_OK;
  return ctx->dtype == QS_C128 ? backward_t<double>(ctx, grads) : backward_t<float>(ctx, grads);
}

int qs_adjoint_stats(const qs_adjoint *ctx, uint64_t *sweeps, uint64_t *kernels) {
  if (!ctx || !sweeps || !kernels) return fail_arg("NULL argument");
  *sweeps = ctx->sweeps;
  *kernels = ctx->kernels;
  return QS_OK;
}

int qs_adjoint_reverse_stats(const qs_adjoint *ctx, uint64_t *blocks, uint64_t *restores) {
  if (!ctx || !blocks || !restores) return fail_arg("NULL argument");
  *blocks = ctx->rev_blocks;
  *restores = ctx->rev_restores;
  return QS_OK;
}

void qs_adjoint_free(qs_adjoint *ctx) { free_ctx(ctx); }

}  // extern "C"
