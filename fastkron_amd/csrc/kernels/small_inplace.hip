// Whole rows of small square factors in one launch (MKM layout, 2 <= P <= 8, any mix, fp32 or fp64): 3^n, 5^n, 6^n,
// 7^n, 8^n with row counts the 8x8 matrix-core kernel does not take, 2x3x5x7 ...
//
// When the factors of a launch cover whole rows, the sliced multiply of all of them leaves every digit of the column
// index where it was, and with square factors also its extent.  The factors are therefore applied in place to rows
// kept in LDS: a pass takes one to three adjacent digits, a thread reads the P^D values of a digit group into
// registers, applies the D factors there and writes the values back to where they came from.  One copy of the rows
// (not two buffers), one barrier per pass, nf / D passes.  Factor values are the same in all lanes and enter the FMAs
// as scalar operands.
//
//   load     one contiguous piece of memory, 16 bytes per lane whatever its alignment: the LDS copy is shifted by
//            the 0 .. 3 elements that the piece starts behind a 16-byte boundary;
//   passes   last digits first; lanes run over the faster digits, the first pass (digit groups contiguous) reads with
//            an odd lane stride (no bank conflicts) or, for even P, with 16-byte accesses;
//   store    straight from the registers of the last pass where its lanes cover runs of 64 elements or more,
//            otherwise from LDS.
//
// Bound: memory in principle.  Two workgroups of 62.5 KB per CU (5^6) that load, multiply and store go through these phases
// with the whole device: 3.9 us of FMAs (9390 cycles by the instruction count) and 5.7 us of memory per row and CU, 37.5 of
// the 44.5 us of sgemkm 1001 x 5^6 one after the other.  Long rows of equal factors therefore have a form of their own
// (kron_rows_inplace_kernel): sgemkm 1001 x 5^6 50.2 -> 38.1 us (3.3 TB/s; cold operands), 8192 x 5^6 322 -> 237 (4.3), 1001 x 7^5
// 62.9 -> 52.5, 4096 x 5^5 31.7 -> 24.8, dgemkm 1001 x 3^8 33.3 -> 23.3 (4.5), 1001 x 6^5 51.6 -> 30.0, 700 x 7^5 98 -> 70.
// Measured against two launches of the kernel with two LDS buffers and one factor per pass (fused_small.hip): sgemkm
// 1001 x 5^6 90.6 -> 44.5 us, 4096 x 5^5 62.4 -> 28.6, 1000 x 7^5 128 -> 58, dgemkm 1000 x 3^8 89 -> 28, 1000 x 6^5 112 -> 48.
// Tried and slower: the next tile's pieces in registers in the general kernel (45 -> 53 us: its passes of every width leave
// no registers, 60 spilled); a start delay of a CU's second workgroup, in either form (3 us: 43.4 -> 45.9); 5^6 in passes of
// three digits, 128 threads per row (1 row 9.5 -> 12.7 us, 8192 rows 237 -> 259; 1001 rows 43.4 -> 40.6).
// The reference fuses factors in shared memory between two buffers (reference src/kernels/cuda/kernel.cuh:165-219).
#include <hip/hip_runtime.h>
#include <algorithm>
#include <type_traits>
#include "../problem.h"
#include "launch.h"

namespace fk {

constexpr uint32_t kIpMaxP = 8;
constexpr uint32_t kIpMaxThreads = 640;      // 625 digit groups of 5^6 in one round
constexpr size_t kIpLdsMax = 160 * 1024;

struct InplacePass { uint32_t f0, p, d, s, magic; };     // factors f0 .. f0+d-1, distance s between values of the first
struct InplaceTile {
  uint32_t P, K, rows, passes, direct, threads, tiles;            // P: of all factors, 0 if they differ
  InplacePass ps[kMaxFused];
};

constexpr int ipPow(int p, int d) { return d == 0 ? 1 : p * ipPow(p, d - 1); }

// out = alpha * v (+ beta * y)
template <typename T, bool HAS_Y>
struct IpOut {
  T* out; const T* y; T alpha, beta;
  __amdgpu_buffer_rsrc_t target, yTarget;                    // the same as buffer descriptors
  // columns: the operand as well, byte offsets of the lane's column in the three, bytes from a row to the next
  __amdgpu_buffer_rsrc_t source;
  uint32_t laneIn, laneOut, laneY, pitch;
  __device__ __forceinline__ void put(uint32_t e, T v) const {
    v *= alpha;
    if (HAS_Y) v += beta * y[e];
    out[e] = v;
  }
};

// S: the distance between the values of the fastest digit when it is known at compile time (the values' addresses are
// then offsets of one register), 0 otherwise.
// SYNC: a barrier behind the reads of the values (one digit group per thread at most): the rows' LDS is free from there on.
// TU: 0 for rows; columns otherwise, so many in LDS next to each other, read from memory by the first pass (FIRST).
template <typename T, int P, int D, int S, bool HAS_Y, bool SYNC = false, bool ST = false, int TU = 0, bool FIRST = false>
__device__ __forceinline__ void ipPass(T* __restrict__ rows, const KernelArgs& a, const InplacePass& ps, const uint32_t b,
                                       const uint32_t E, const bool vec, const bool toMemory, const IpOut<T, HAS_Y>& o) {
  constexpr int N = ipPow(P, D), VE = 16 / (int)sizeof(T);
  constexpr int U = N >= 16 ? 1 : N >= 6 ? 2 : 4;            // digit groups per thread and round
  constexpr int kScalars = D == 3 ? 75 : D == 2 && P == 6 && sizeof(T) == 8 ? 72 : 64;                 // scalar registers for factor values
  constexpr bool kHoist = D * P * P * (int)sizeof(T) / 4 <= kScalars;
  constexpr int TQ0 = kScalars * 4 / (int)sizeof(T) / P, TQ = TQ0 < P ? TQ0 : P;      // columns of a factor at a time
  static_assert(TQ == P || D == 1, "the values read are overwritten after all columns");
  typedef T VT __attribute__((ext_vector_type(VE)));
  typedef const __attribute__((address_space(4))) T* ConstPtr;
  static_assert(!SYNC || U == 1, "one group per thread");
  const uint32_t s = S ? S : ps.s, groups = E / N, nth = blockDim.x;
  uint32_t tid = threadIdx.x;
  if (SYNC) asm volatile("" : "+v"(tid));                     // (what depends on it would be kept in registers from tile to tile)
  // (read-only for the whole launch, the same address in every lane: the constant address space makes these scalar loads)
  auto loadF = [&](int d, int q0, T (&F_)[P][TQ]) {
    uint64_t fa = (uint64_t)((const T*)a.f[ps.f0 + d] + (size_t)b * a.f_batch[ps.f0 + d]);
    if (!kHoist) {
      // all factor values of a pass do not fit the scalar registers: opaque, so that they are not kept for the next round
      asm volatile("" : "+s"(fa));
      __builtin_amdgcn_sched_barrier(0);
    }
    const ConstPtr F = (ConstPtr)(uintptr_t)fa;
    // (a factor is stored P x P one way or the other: constant offsets become wide scalar loads)
    const bool pMajor = a.f_sq[ps.f0 + d] == 1;
    if constexpr (TQ == P) {
      // (selected as whole numbers: selections of floating-point values would move them to vector registers)
      typedef std::conditional_t<sizeof(T) == 4, uint32_t, uint64_t> W;
      W m[P * P];
#pragma unroll
      for (int i = 0; i < P * P; i++) m[i] = __builtin_bit_cast(W, (T)F[i]);
#pragma unroll
      for (int p = 0; p < P; p++)
#pragma unroll
        for (int q = 0; q < P; q++) F_[p][q] = __builtin_bit_cast(T, p == q || pMajor ? m[p * P + q] : m[q * P + p]);
    } else if (pMajor) {
#pragma unroll
      for (int p = 0; p < P; p++)
#pragma unroll
        for (int q = 0; q < TQ; q++) if (q0 + q < P) F_[p][q] = F[p * P + q0 + q];
    } else {
#pragma unroll
      for (int q = 0; q < TQ; q++)
#pragma unroll
        for (int p = 0; p < P; p++) if (q0 + q < P) F_[p][q] = F[p + (q0 + q) * P];
    }
  };
  T Fk[kHoist ? D : 1][P][TQ];
  if constexpr (kHoist) {
#pragma unroll
    for (int d = 0; d < D; d++) loadF(d, 0, Fk[d]);
  }
  for (uint32_t g0 = tid; SYNC ? g0 < nth : g0 < groups; g0 += U * nth) {
    uint32_t step = s;
    asm volatile("" : "+s"(step));                             // (its multiples would fill the registers)
    uint32_t e0[U];
    T x[U][N];
    const bool v16 = S == 1 && N % VE == 0 && vec;
#pragma unroll
    for (int k = 0; k < U; k++) {
      const uint32_t g = g0 + k * nth;
      const uint32_t hi = S == 1 ? g : S ? g / (uint32_t)(S ? S : 1) : __umulhi(g, ps.magic);
      e0[k] = hi * (s * N) + (g - hi * s);
      if ((U > 1 || SYNC) && g >= groups) continue;
      if constexpr (FIRST) {
        const uint32_t lane = o.laneIn + e0[k] / (TU ? TU : 1) * o.pitch, row = step / (TU ? TU : 1) * o.pitch;
#pragma unroll
        for (uint32_t i = 0; i < N; i++) x[k][i] = bufferLoad<T>(o.source, lane, i * row);
      } else if (v16) {
#pragma unroll
        for (int i = 0; i < N / VE; i++) {
          const VT t = *(const VT*)(rows + e0[k] + i * VE);
#pragma unroll
          for (int j = 0; j < VE; j++) x[k][i * VE + j] = t[j];
        }
      } else {
        uint32_t at = e0[k];
#pragma unroll
        for (int i = 0; i < N; i++, at += step) x[k][i] = rows[S ? e0[k] + i * S : at];
      }
    }
    if (SYNC) __syncthreads();
#pragma unroll
    for (int d = 0; d < D; d++) {
      const int st = ipPow(P, d);
      T u[TQ == P ? 1 : U][TQ == P ? 1 : P];
      if constexpr (TQ < P) {
#pragma unroll
        for (int k = 0; k < U; k++)
#pragma unroll
          for (int p = 0; p < P; p++) u[k][p] = x[k][p];
      }
#pragma unroll
      for (int q0 = 0; q0 < P; q0 += TQ) {
        T Fl[P][TQ];
        if constexpr (!kHoist) loadF(d, q0, Fl);
#pragma unroll
        for (int k = 0; k < U; k++)
#pragma unroll
          for (int r = 0; r < N / P; r++) {
            const int i0 = r / st * (st * P) + r % st;
            T v[P];
#pragma unroll
            for (int p = 0; p < P; p++) v[p] = TQ < P ? u[TQ == P ? 0 : k][TQ == P ? 0 : p] : x[k][i0 + p * st];
#pragma unroll
            for (int q = 0; q < TQ; q++) {
              if (q0 + q >= P) continue;
              T acc = v[0] * (kHoist ? Fk[kHoist ? d : 0][0][q] : Fl[0][q]);
#pragma unroll
              for (int p = 1; p < P; p++) acc += v[p] * (kHoist ? Fk[kHoist ? d : 0][p][q] : Fl[p][q]);
              x[k][i0 + (q0 + q) * st] = acc;
            }
          }
      }
    }
#pragma unroll
    for (int k = 0; k < U; k++) {
      if ((U > 1 || SYNC) && g0 + k * nth >= groups) continue;
      uint32_t at = e0[k];
      if (toMemory) {
        // through buffer descriptors: one address register per group, the values' distances as scalar offsets
        const uint32_t row = TU ? e0[k] / (TU ? TU : 1) * o.pitch : 0, next = TU ? step / (TU ? TU : 1) * o.pitch : 0;
        T yv[HAS_Y ? N : 1];
        if constexpr (HAS_Y) {
#pragma unroll
          for (uint32_t i = 0; i < N; i++)
            yv[i] = TU ? bufferLoad<T>(o.yTarget, o.laneY + row, i * next) : bufferLoad<T>(o.yTarget, e0[k] * sizeof(T), i * step * sizeof(T));
        }
#pragma unroll
        for (uint32_t i = 0; i < N; i++) {
          T v = x[k][i] * o.alpha;
          if constexpr (HAS_Y) v += o.beta * yv[i];
          if (TU) bufferStore<ST>(v, o.target, o.laneOut + row, i * next);
          else bufferStore<ST>(v, o.target, e0[k] * sizeof(T), i * step * sizeof(T));
        }
      } else if (v16) {
#pragma unroll
        for (int i = 0; i < N / VE; i++) {
          VT t;
#pragma unroll
          for (int j = 0; j < VE; j++) t[j] = x[k][i * VE + j];
          *(VT*)(rows + e0[k] + i * VE) = t;
        }
      } else {
#pragma unroll
        for (int i = 0; i < N; i++, at += step) rows[S ? e0[k] + i * S : at] = x[k][i];
      }
    }
  }
}

// The pass with its distance as a constant where the chain is one of equal factors (1, P^D, P^2D) or begins it.
template <typename T, int P, int D, bool HAS_Y>
__device__ __forceinline__ void ipPassAny(T* __restrict__ rows, const KernelArgs& a, const InplacePass& ps, const uint32_t b,
                                          const uint32_t E, const bool vec, const bool toMemory, const IpOut<T, HAS_Y>& o) {
  constexpr int N = ipPow(P, D);
  if (ps.s == 1) return ipPass<T, P, D, 1, HAS_Y>(rows, a, ps, b, E, vec, false, o);
  if constexpr (N >= 25) {
    if (ps.s == N) return ipPass<T, P, D, N, HAS_Y>(rows, a, ps, b, E, false, toMemory, o);
    if constexpr (P < 7) { if (ps.s == N * N) return ipPass<T, P, D, N * N, HAS_Y>(rows, a, ps, b, E, false, toMemory, o); }
  }
  ipPass<T, P, D, 0, HAS_Y>(rows, a, ps, b, E, false, toMemory, o);
}

// Digits per pass: as many as their values fit the registers.
constexpr int ipDepth(int p, size_t es) { return p <= 3 ? 3 : p <= 5 || (p <= 7 && es == 4) ? 2 : 1; }
// Waves per SIMD: fp32 rows of up to 80 KB run as two workgroups of ten waves per CU; the wider groups have fewer
// threads (6^5: 216 groups, 7^5: 343) and take more registers.
constexpr int ipWaves(int p, size_t es) { return es == 8 || p == 7 ? 3 : p == 6 || p == 8 || p == 0 ? 4 : 5; }

// P: all factors are PxP; 0: any mix, one digit per pass.
template <typename T, int P, bool HAS_Y>
__global__ __launch_bounds__(kIpMaxThreads, ipWaves(P, sizeof(T)))
void kron_small_inplace_kernel(const KernelArgs a, const InplaceTile t, const OuterStrides outer) {
  constexpr uint32_t VE = 16 / sizeof(T);
  typedef T VT __attribute__((ext_vector_type(VE)));
  extern __shared__ __align__(16) unsigned char ipLds[];
  const uint32_t tid = threadIdx.x, nth = blockDim.x, b = blockIdx.y;
  const uint32_t m0 = blockIdx.x * t.rows;
  const uint32_t E = (a.M - m0 < t.rows ? a.M - m0 : t.rows) * t.K;
  const T* src = (const T*)a.in + (size_t)b * a.in_batch + (size_t)blockIdx.z * outer.in + (size_t)m0 * t.K;
  const uint32_t shift = (uint32_t)((uintptr_t)src / sizeof(T)) & (VE - 1);
  VT* chunks = (VT*)ipLds;
  T* rows = (T*)ipLds + shift;
  IpOut<T, HAS_Y> o;
  o.out = (T*)a.out + (size_t)b * a.out_batch + (size_t)blockIdx.z * outer.out + (size_t)m0 * t.K;
  o.y = HAS_Y ? (const T*)a.y + (size_t)b * a.y_batch + (size_t)blockIdx.z * outer.y + (size_t)m0 * t.K : nullptr;
  o.target = streamTarget(o.out, E * (uint32_t)sizeof(T));
  if (HAS_Y) o.yTarget = streamTarget((void*)o.y, E * (uint32_t)sizeof(T));
  o.alpha = a.epilogue ? (T)a.alpha : T(1); o.beta = (T)a.beta;

  // 16-byte pieces that lie inside the rows, then the elements before the first and behind the last of them
  const uint32_t first = shift ? 1 : 0, last = (shift + E) / VE;
  constexpr int LU = 8;
  for (uint32_t c0 = first + tid; c0 < last; c0 += LU * nth) {
    VT v[LU];
#pragma unroll
    for (int k = 0; k < LU; k++) if (c0 + k * nth < last) v[k] = *(const VT*)(src + ((int64_t)(c0 + k * nth) * VE - shift));
#pragma unroll
    for (int k = 0; k < LU; k++) if (c0 + k * nth < last) chunks[c0 + k * nth] = v[k];
  }
  if (tid < 2 * VE) {
    const uint32_t e = tid < VE ? tid : E - 1 - (tid - VE);
    if (e < E) {
      const uint32_t c = (shift + e) / VE;
      if (c < first || c >= last) rows[e] = src[e];
    }
  }
  __syncthreads();

  for (uint32_t i = 0; i < t.passes; i++) {
    const InplacePass ps = t.ps[i];
    const bool toMemory = t.direct && i + 1 == t.passes;
    if constexpr (P == 0) {
      switch (ps.p) {
#define IP_CASE(PV) case PV: ipPassAny<T, PV, 1, HAS_Y>(rows, a, ps, b, E, shift == 0, toMemory, o); break;
        IP_CASE(2) IP_CASE(3) IP_CASE(4) IP_CASE(5) IP_CASE(6) IP_CASE(7) IP_CASE(8)
#undef IP_CASE
        default: break;
      }
    } else {
      constexpr int D = ipDepth(P, sizeof(T));
      if (ps.d == D) ipPassAny<T, P, D, HAS_Y>(rows, a, ps, b, E, shift == 0, toMemory, o);
      else if (ps.d == 1) ipPassAny<T, P, 1, HAS_Y>(rows, a, ps, b, E, shift == 0, toMemory, o);
      else if constexpr (D == 3) ipPassAny<T, P, 2, HAS_Y>(rows, a, ps, b, E, shift == 0, toMemory, o);
    }
    if (!toMemory) __syncthreads();
  }
  if (t.direct) return;

  const bool v16 = shift == 0 && (uintptr_t)o.out % 16 == 0 && (!HAS_Y || (uintptr_t)o.y % 16 == 0);
  const uint32_t whole = v16 ? E / VE : 0;
  for (uint32_t c = tid; c < whole; c += nth) {
    VT v = chunks[c] * o.alpha;
    if (HAS_Y) v += ((const VT*)o.y)[c] * o.beta;
    ((VT*)o.out)[c] = v;
  }
  for (uint32_t e = whole * VE + tid; e < E; e += nth) o.put(e, rows[e]);
}

struct InplaceNoOuter {};
struct InplaceOuter { OuterStrides outer; uint32_t inner; };

// Rows of NF equal factors, one row per workgroup at a time and as many workgroups as the device holds at once: the next
// row's pieces are on their way to registers while this one's digits are multiplied, and go to LDS as soon as the last pass
// has read its values (its stores follow).
template <int P, int NF, size_t ES> struct IpRow {
  static constexpr int VE = 16 / (int)ES, K = ipPow(P, NF);
  // digits per pass (two of 6 in fp64 need the next factor's values after the first's; two of 7 do not fit); what is left over
  // is the first pass, so that the last one is wide
  static constexpr int D = P <= 3 ? 3 : P == 7 && ES == 8 ? 1 : 2, N = ipPow(P, D), R = NF % D ? NF % D : D;
  static constexpr int groups = K / N, threads = groups <= (int)kIpMaxThreads ? (groups + 63) / 64 * 64 : (int)kIpMaxThreads;
  static constexpr bool oneRound = groups <= threads;
  static constexpr int loads = (K / VE + 1 + threads - 1) / threads;             // 16-byte pieces per thread
  // workgroups per CU: by LDS, and by the registers of the values, of the pieces and of the rest
  static constexpr int regs = N * (oneRound ? 1 : 2) * (int)ES / 4 + 4 * loads + 40;
  static constexpr int byLds = (int)kIpLdsMax / (K * (int)ES + 16), byRegs = 4 * (512 / ((regs + 7) / 8 * 8)) / (threads / 64);
  static constexpr int perCU = byLds < byRegs ? byLds : byRegs, waves = (perCU * threads / 64 + 3) / 4;
};

template <typename T, int P, int NF, int J, bool HAS_Y, bool ST>
__device__ __forceinline__ void ipRowPasses(T* rows, const KernelArgs& a, const uint32_t b, const bool vec, const IpOut<T, HAS_Y>& o) {
  using C = IpRow<P, NF, sizeof(T)>;
  constexpr int F0 = J == 0 ? 0 : C::R + (J - 1) * C::D, D = J == 0 ? C::R : C::D;
  constexpr bool last = F0 + D == NF;
  InplacePass ps{};
  ps.f0 = F0; ps.p = P; ps.d = D; ps.s = ipPow(P, F0);
  asm volatile("" : "+s"(ps.f0));                              // (factor values of the next row are not this row's to keep)
  ipPass<T, P, D, ipPow(P, F0), HAS_Y, last && C::oneRound, ST>(rows, a, ps, b, C::K, vec, last, o);
  if constexpr (!last || !C::oneRound) __syncthreads();
  if constexpr (!last) {
    ipRowPasses<T, P, NF, J + 1, HAS_Y, ST>(rows, a, b, vec, o);
  }
}

// NT: 0 ordinary accesses, 1 non-temporal loads, 2 non-temporal loads and stores.  OUTER: two batch dimensions (asked for at run
// time, the second one cost the form with one of them 1 us of 37, 1001 x 5^6 fp32).
template <typename T, int P, int NF, bool HAS_Y, int NT, bool OUTER>
__global__ __launch_bounds__((IpRow<P, NF, sizeof(T)>::threads), (IpRow<P, NF, sizeof(T)>::waves))
void kron_rows_inplace_kernel(const KernelArgs a, const uint32_t total, const std::conditional_t<OUTER, InplaceOuter, InplaceNoOuter> two) {
  using C = IpRow<P, NF, sizeof(T)>;
  constexpr uint32_t VE = C::VE, K = C::K;
  typedef T VT __attribute__((ext_vector_type(C::VE)));
  extern __shared__ __align__(16) unsigned char ipLds[];
  VT* chunks = (VT*)ipLds;
  IpOut<T, HAS_Y> o;
  o.alpha = a.epilogue ? (T)a.alpha : T(1); o.beta = (T)a.beta;

  // 16-byte pieces that lie inside the row, and the elements before the first and behind the last of them
  struct Row { const T* src; uint32_t b, o, m, shift, last; };
  auto rowAt = [&](uint32_t i) {
    Row r;
    r.b = a.batch == 1 ? 0 : i / a.M; r.m = i - r.b * a.M; r.o = 0;
    if constexpr (OUTER) { r.o = r.b / two.inner; r.b -= r.o * two.inner; }
    r.src = (const T*)a.in + (size_t)r.b * a.in_batch + (size_t)r.m * K;
    if constexpr (OUTER) r.src += (size_t)r.o * two.outer.in;
    r.shift = (uint32_t)((uintptr_t)r.src / sizeof(T)) & (VE - 1);
    r.last = (r.shift + K) / VE;
    return r;
  };
  VT v[C::loads];
  T edge = T(0);
  auto edgeOf = [&](const Row& r, uint32_t tid, uint32_t* e) {
    const uint32_t behind = r.last * VE - r.shift;             // first element behind the last piece
    *e = tid < VE ? tid : behind + tid - VE;
    return tid < 2 * VE && (tid < VE ? r.shift != 0 && tid < VE - r.shift : *e < K);
  };
  auto fetch = [&](const Row& r) {
    uint32_t tid = threadIdx.x, e;
    asm volatile("" : "+v"(tid));
    // (beyond `last`, and piece 0 where it begins before the row: outside the descriptor's range, nothing is read)
    const auto from = streamTarget((void*)(r.src - r.shift), r.last * 16);
    if (edgeOf(r, tid, &e)) edge = r.src[e];
    const uint32_t off = tid * 16;
#pragma unroll
    for (int k = 0; k < C::loads; k++)
      v[k] = __builtin_bit_cast(VT, __builtin_amdgcn_raw_buffer_load_b128(from, (int)(k == 0 && tid == 0 && r.shift ? 0x7ffffff0u : off),
                                                                         k * C::threads * 16, NT ? 2 : 0));
  };

  uint32_t i = blockIdx.x;
  Row r = rowAt(i);
  fetch(r);
  for (;;) {
    T* rows = (T*)ipLds + r.shift;
    const uint32_t b = r.b;
    o.out = (T*)a.out + (size_t)b * a.out_batch + (size_t)r.m * K;
    o.y = HAS_Y ? (const T*)a.y + (size_t)b * a.y_batch + (size_t)r.m * K : nullptr;
    if constexpr (OUTER) {
      o.out += (size_t)r.o * two.outer.out;
      if (HAS_Y) o.y += (size_t)r.o * two.outer.y;
    }
    o.target = streamTarget(o.out, K * (uint32_t)sizeof(T));
    if (HAS_Y) o.yTarget = streamTarget((void*)o.y, K * (uint32_t)sizeof(T));
    {
      uint32_t tid = threadIdx.x, e;
      asm volatile("" : "+v"(tid));
#pragma unroll
      for (int k = 0; k < C::loads; k++) {
        const uint32_t c = tid + k * C::threads;
        if ((k > 0 || c > 0 || r.shift == 0) && ((k + 1) * C::threads <= (int)(K / VE) || c < r.last)) chunks[c] = v[k];
      }
      if (edgeOf(r, tid, &e)) rows[e] = edge;
    }
    __syncthreads();
    const bool vec = r.shift == 0, more = i + gridDim.x < total;
    if (more) {
      i += gridDim.x;
      r = rowAt(i);
      fetch(r);
    }
    ipRowPasses<T, P, NF, 0, HAS_Y, NT == 2>(rows, a, b, vec, o);
    if (!more) return;
  }
}

// Columns (KMM layout): all K = P^NF rows of TU neighbouring columns per workgroup.  Batch entries that share the factors
// count as further columns, so that a few columns per entry fill the lanes as well.  The first pass reads its values from
// memory, the last one writes its results there, lanes along the columns; LDS holds the values in between (none with a single
// pass).  Bound: memory; 128 bytes of a row per access, the digits of one or two passes as independent loads per lane.
// TU is 32 (fp32) and 16 (fp64, 32 for short columns): 44 to 80 KB of LDS, two or three workgroups per CU.
// Chains of GeKMM run as groups of such launches with their digits left where they are (Handle::runColumns), us before (one
// plain launch per factor, groups of the kernel with two LDS buffers, or fp64 factors merged to 64x64) -> after: sgekmm
// 7^6 x 88 117 -> 55 (2 x 1.5 TB/s), 7^5 x 1024 132 -> 61, 5^6 x 1024 115 -> 54, 3^8 x 1024 67 -> 29, 8^5 x 88 27.6 -> 21,
// dgekmm 8^5 x 88 88 -> 31, 8^3 x 787, 12 entries 76 -> 33, 6^6 x 300 237 -> 101, 5^4 x 1024 18 -> 7.
template <int P, int NF, size_t ES, bool NARROW> struct IpCols {
  static constexpr int K = ipPow(P, NF);
  static constexpr int most = P == 2 ? (ES == 4 ? 6 : 3) : P == 3 ? 3 : P == 4 ? (ES == 4 ? 3 : 2) : P <= 6 || ES == 4 ? 2 : 1;
  static constexpr int passes = (NF + most - 1) / most, D = (NF + passes - 1) / passes, N = ipPow(P, D);      // digits of every pass but the last
  static constexpr int U = N >= 16 ? 1 : N >= 6 ? 2 : 4;
  static constexpr int TU = passes == 1 ? 64 : NARROW ? 8 : K * 32 * (int)ES <= (ES == 4 ? 81920 : 49152) ? 32 : 16;
  static constexpr int groups = K / N * TU, threads0 = ((groups + U - 1) / U + 63) / 64 * 64, threads = threads0 < 512 ? threads0 : 512;
  static constexpr int lds = passes == 1 ? 0 : K * TU * (int)ES;
  static constexpr int regs = N * U * (int)ES / 4 + (N >= 64 ? 90 : 48), byRegs = 512 / ((regs + 7) / 8 * 8);
  static constexpr int perCU = passes == 1 ? 32 : (int)kIpLdsMax / lds, waves0 = (perCU * threads / 64 + 3) / 4;
  static constexpr int waves1 = waves0 < byRegs ? waves0 : byRegs, waves = waves1 > 8 ? 8 : waves1;
};

template <typename T, int P, int NF, int F0, bool HAS_Y, bool NARROW>
__device__ __forceinline__ void ipColPasses(T* cols, const KernelArgs& a, const uint32_t b, const IpOut<T, HAS_Y>& o) {
  using C = IpCols<P, NF, sizeof(T), NARROW>;
  constexpr int D = NF - F0 < C::D ? NF - F0 : C::D;
  constexpr bool last = F0 + D == NF;
  InplacePass ps{};
  ps.f0 = F0; ps.p = P; ps.d = D; ps.s = C::TU * ipPow(P, F0);
  ipPass<T, P, D, C::TU * ipPow(P, F0), HAS_Y, false, false, C::TU, F0 == 0>(cols, a, ps, b, C::K * C::TU, false, last, o);
  if constexpr (!last) {
    __syncthreads();
    ipColPasses<T, P, NF, F0 + D, HAS_Y, NARROW>(cols, a, b, o);
  }
}

template <typename T, int P, int NF, bool HAS_Y, bool NARROW>
__global__ __launch_bounds__((IpCols<P, NF, sizeof(T), NARROW>::threads), (IpCols<P, NF, sizeof(T), NARROW>::waves))
void kron_cols_inplace_kernel(const KernelArgs a, const uint32_t total) {
  using C = IpCols<P, NF, sizeof(T), NARROW>;
  constexpr uint32_t ES = sizeof(T);
  extern __shared__ __align__(16) unsigned char ipLds[];
  // (a grid dimension for entries with factors of their own)
  const uint32_t b = blockIdx.y, u0 = blockIdx.x * C::TU, u = u0 + threadIdx.x % C::TU;
  const uint32_t h0 = u0 / a.M, h = u / a.M, c = u - h * a.M, entries = a.batch / gridDim.y, hEnd = (u0 + C::TU - 1) / a.M;
  const uint32_t more = (hEnd < entries ? hEnd : entries - 1) - h0;             // entries behind the first that the tile reaches
  IpOut<T, HAS_Y> o;
  o.alpha = a.epilogue ? (T)a.alpha : T(1); o.beta = (T)a.beta;
  o.pitch = a.M * ES;
  const bool live = u < total;
  auto lane = [&](uint64_t stride) { return live ? (uint32_t)(((h - h0) * stride + c) * ES) : 0x7ffffff0u; };      // (others: out of range)
  auto range = [&](uint64_t stride) { return (uint32_t)((more * stride + (uint64_t)C::K * a.M) * ES); };
  const uint64_t e0 = (uint64_t)b + h0;
  o.source = streamTarget((T*)a.in + e0 * a.in_batch, range(a.in_batch)); o.laneIn = lane(a.in_batch);
  o.target = streamTarget((T*)a.out + e0 * a.out_batch, range(a.out_batch)); o.laneOut = lane(a.out_batch);
  if (HAS_Y) { o.yTarget = streamTarget((T*)a.y + e0 * a.y_batch, range(a.y_batch)); o.laneY = lane(a.y_batch); }
  ipColPasses<T, P, NF, 0, HAS_Y, NARROW>((T*)ipLds, a, b, o);
}

static bool ipTile(uint32_t nf, const uint32_t* p, const uint32_t* q, uint64_t Kin, uint32_t M, uint32_t batch, DType dt,
                   InplaceTile* t) {
  if (nf < 1 || nf > kMaxFused || M == 0) return false;
  const size_t es = dtypeSize(dt);
  uint64_t K = 1;
  bool mixed = false;
  for (uint32_t j = 0; j < nf; j++) {
    if (p[j] < 2 || p[j] > kIpMaxP || q[j] != p[j]) return false;
    K *= p[j];
    if (p[j] != p[0]) mixed = true;
  }
  if (K != Kin || K * es + 16 > kIpLdsMax) return false;
  *t = InplaceTile{};
  t->K = (uint32_t)K; t->P = mixed ? 0 : p[0];
  // several short rows per workgroup: up to 32 KB while that leaves two workgroups per CU and more
  t->rows = 1;
  while (2 * t->rows * K * es <= 32768 && (uint64_t)M * batch / (2 * t->rows) >= 512) t->rows *= 2;
  t->tiles = (M + t->rows - 1) / t->rows;
  uint32_t s = 1, widest = 1;
  for (uint32_t j = 0; j < nf;) {
    InplacePass& ps = t->ps[t->passes++];
    const uint32_t dmax = mixed ? 1 : ipDepth(p[j], es);
    uint32_t d = 1, n = p[j];
    while (d < dmax && j + d < nf && p[j + d] == p[j]) { d++; n *= p[j]; }
    ps.f0 = j; ps.p = p[j]; ps.d = d; ps.s = s;
    // floor(g / s) = mulhi(g, magic) for g * s < 2^32: g and s are below the rows' element count, at most 40960, over n
    ps.magic = s == 1 ? 0 : (uint32_t)((1ull << 32) / s) + 1;
    const uint32_t groups = (uint32_t)(t->rows * K / n);
    if (groups > widest) widest = groups;
    j += d;
    t->direct = s >= 64;
    s *= n;
  }
  // One group per thread; with enough tiles to fill the device rather 256 threads (and more rounds) than fewer workgroups
  // per CU than their LDS allows.
  uint32_t most = kIpMaxThreads;
  if ((uint64_t)t->tiles * batch >= 512) {
    const uint32_t perCU = (uint32_t)(kIpLdsMax / (t->rows * K * es + 16));
    const uint32_t fit = 64 * (4 * ipWaves(t->P, es) / perCU);
    most = fit > kIpMaxThreads ? kIpMaxThreads : fit < 256 ? 256 : fit;
  }
  const uint32_t rounds = (widest + most - 1) / most;
  t->threads = ((widest + rounds - 1) / rounds + 63) / 64 * 64;
  return true;
}

bool smallInplaceFits(uint32_t nf, const uint32_t* p, const uint32_t* q, uint64_t Kin, uint32_t M, uint32_t batch, DType dt) {
  InplaceTile t;
  return ipTile(nf, p, q, Kin, M, batch, dt, &t);
}

bool smallInplaceSupported(const StepArgs& a, DType dt) {
  if (a.batch == 0 || a.batch > 65535 || a.Kin != a.Kout) return false;
  if (a.in_ldc != 1 || a.out_ldc != 1 || a.in_ldm != (int64_t)a.Kin || a.out_ldm != (int64_t)a.Kin) return false;
  if (a.y && (a.y_ldc != 1 || a.y_ldm != (int64_t)a.Kin)) return false;
  for (uint32_t j = 0; j < a.nf && j < kMaxFused; j++)
    if (!(a.f_sq[j] == 1 && a.f_sp[j] == (int64_t)a.q[j]) && !(a.f_sp[j] == 1 && a.f_sq[j] == (int64_t)a.p[j])) return false;
  return smallInplaceFits(a.nf, a.p, a.q, a.Kin, a.M, a.batch, dt);
}

template <typename T, int P, bool HAS_Y>
static hipError_t launchIpP(const StepArgs& a, const InplaceTile& t, hipStream_t stream) {
  static PerDeviceOnce attrOnce;
  const int dev = launchDeviceIndex();
  const size_t lds = (size_t)t.rows * t.K * sizeof(T) + 16;
  if (lds > 65536 && !attrOnce.done(dev)) {
    hipError_t e = hipFuncSetAttribute((const void*)kron_small_inplace_kernel<T, P, HAS_Y>, hipFuncAttributeMaxDynamicSharedMemorySize,
                                       (int)kIpLdsMax);
    if (e != hipSuccess) return e;
    attrOnce.mark(dev);
  }
  hipLaunchKernelGGL((kron_small_inplace_kernel<T, P, HAS_Y>), dim3(t.tiles, innerEntries(a), outerEntries(a)), dim3(t.threads), lds,
                     stream, a, t, a.outer);
  return hipGetLastError();
}

template <typename T>
static hipError_t launchIpT(const StepArgs& a, const InplaceTile& t, hipStream_t stream) {
  const bool y = a.y && a.epilogue;
  switch (t.P) {
#define IP_CASE(P) case P: return y ? launchIpP<T, P, true>(a, t, stream) : launchIpP<T, P, false>(a, t, stream);
    IP_CASE(0) IP_CASE(2) IP_CASE(3) IP_CASE(4) IP_CASE(5) IP_CASE(6) IP_CASE(7) IP_CASE(8)
#undef IP_CASE
    default: return hipErrorInvalidValue;
  }
}

template <typename T, int P, int NF, bool HAS_Y, int NT, bool OUTER>
static hipError_t launchIpRowsAs(const StepArgs& a, uint32_t total, uint32_t grid, hipStream_t stream) {
  using C = IpRow<P, NF, sizeof(T)>;
  static PerDeviceOnce attrOnce;
  const int dev = launchDeviceIndex();
  const auto kernel = kron_rows_inplace_kernel<T, P, NF, HAS_Y, NT, OUTER>;
  const size_t lds = C::K * sizeof(T) + 16;
  if (lds > 65536 && !attrOnce.done(dev)) {
    if (const hipError_t e = hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)kIpLdsMax); e != hipSuccess) return e;
    attrOnce.mark(dev);
  }
  if constexpr (OUTER) hipLaunchKernelGGL(kernel, dim3(grid), dim3(C::threads), lds, stream, a, total, InplaceOuter{a.outer, a.inner});
  else hipLaunchKernelGGL(kernel, dim3(grid), dim3(C::threads), lds, stream, a, total, InplaceNoOuter{});
  return hipGetLastError();
}

// One row per workgroup at a time, if that is the better form (*taken).  Rows per workgroup slot of the device decide:
//   against several workgroups that each take a row and end (kron_small_inplace_kernel): better up to 6 rows per slot for every
//   size (5^5 fp32, 2.7 rows 44.6 -> 37, 8 rows 103 / 109 us; 3^8 fp64, 5 rows 103 -> 92, 13 rows 211 / 216), beyond that where
//   a CU holds one or two rows (5^6 fp32, 16 rows 322 -> 237) or where this form takes more digits per pass or more registers
//   per thread than that kernel (6 and 7: 6^5 fp64, 16 rows 307 -> 220; 7^4 fp32, 13 rows 193 -> 162);
//   streamed operands: non-temporal loads up to 6 rows per slot (4096 x 5^5 fp32 28.0 -> 23.8; beyond 207 / 215), and stores up
//   to 2 (1001 x 5^6 40.5 -> 38.0, 1001 x 6^5 fp64 33.0 -> 30.0; 7000 x 5^5, 2.7 rows 37 / 45: the runs of a wave begin and end
//   inside lines, whose other parts come later the further the workgroups of a CU have drifted apart).
template <typename T, int P, int NF>
static hipError_t launchIpRows(const StepArgs& a, hipStream_t stream, bool* taken) {
  using C = IpRow<P, NF, sizeof(T)>;
  const uint32_t total = a.M * a.batch, resident = (uint32_t)(C::perCU * deviceCUs()), grid = std::min(total, resident);
  *taken = P >= 6 || C::perCU <= 2 || total / 6 <= resident;
  if (!*taken) return hipSuccess;
  const int nt = streamMode(a) < 2 || total / 6 > resident ? 0 : total / 2 > resident ? 1 : 2;
  const bool y = a.y && a.epilogue;
#define IP_ROWS(NT, OUTER) y ? launchIpRowsAs<T, P, NF, true, NT, OUTER>(a, total, grid, stream) : launchIpRowsAs<T, P, NF, false, NT, OUTER>(a, total, grid, stream)
  if (a.inner) return nt == 0 ? IP_ROWS(0, true) : IP_ROWS(1, true);
  return nt == 0 ? IP_ROWS(0, false) : nt == 1 ? IP_ROWS(1, false) : IP_ROWS(2, false);
#undef IP_ROWS
}

// The sizes of rows of equal factors that have the form above: of those of 9 to 160 KB (below, several rows per workgroup fill its
// threads better) the ones that were measured in it; fp64 rows of 3^7, 6^4 and 7^4 (10 to 19 KB) were not and stay with the general
// kernel.  3^9 is more factors than a launch takes.
static hipError_t launchIpRowsAny(const StepArgs& a, const InplaceTile& t, DType dt, hipStream_t stream, bool* taken) {
  *taken = false;
  if ((uint64_t)a.M * a.batch >= (1ull << 31)) return hipSuccess;
  const uint32_t size = t.P * 16 + a.nf;
#define IP_ROWS(T, P, NF) case P * 16 + NF: return launchIpRows<T, P, NF>(a, stream, taken);
  if (dt == DType::F32) switch (size) {
    IP_ROWS(float, 3, 8) IP_ROWS(float, 5, 5) IP_ROWS(float, 5, 6) IP_ROWS(float, 6, 5) IP_ROWS(float, 7, 4) IP_ROWS(float, 7, 5)
    default: return hipSuccess;
  }
  switch (size) {
    IP_ROWS(double, 3, 8) IP_ROWS(double, 5, 5) IP_ROWS(double, 5, 6) IP_ROWS(double, 6, 5) IP_ROWS(double, 7, 5)
    default: return hipSuccess;
  }
#undef IP_ROWS
}

// ---- columns ----
template <typename T, int P, int NF, bool NARROW>
static hipError_t launchIpColsAs(const StepArgs& a, hipStream_t stream) {
  using C = IpCols<P, NF, sizeof(T), NARROW>;
  static PerDeviceOnce attrOnce;
  const int dev = launchDeviceIndex();
  const bool own = a.batch > 1 && a.f_batch[0] != 0, y = a.y && a.epilogue;
  const uint32_t total = own ? a.M : a.M * a.batch;
  if (C::lds > 65536 && !attrOnce.done(dev)) {
    for (const void* k : {(const void*)kron_cols_inplace_kernel<T, P, NF, true, NARROW>, (const void*)kron_cols_inplace_kernel<T, P, NF, false, NARROW>})
      if (const hipError_t e = hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize, (int)kIpLdsMax); e != hipSuccess) return e;
    attrOnce.mark(dev);
  }
  const dim3 grid((total + C::TU - 1) / C::TU, own ? a.batch : 1);
  if (y) hipLaunchKernelGGL((kron_cols_inplace_kernel<T, P, NF, true, NARROW>), grid, dim3(C::threads), C::lds, stream, a, total);
  else hipLaunchKernelGGL((kron_cols_inplace_kernel<T, P, NF, false, NARROW>), grid, dim3(C::threads), C::lds, stream, a, total);
  return hipGetLastError();
}

template <typename T, int P, int NF>
static hipError_t launchIpCols(const StepArgs& a, hipStream_t stream) {
  using C = IpCols<P, NF, sizeof(T), false>;
  // Fewer than one tile for every second CU: 8 columns per workgroup spread them over four (two) times as many (sgekmm 8^5 x 2
  // 25.4 -> 15.4 us, 7^6 x 2 17.8 -> 13.0, 5^8 x 5 29 -> 24, dgekmm 8^6 x 2 20.9 -> 18.7); with more, pieces of 32 and 64 bytes
  // cost more than idle CUs (sgekmm 7^6 x 16 17.9 / 22.3, 6^6 x 24 12.8 / 16.5, 5^8 x 10 29 / 38).
  if constexpr (C::K >= 200) {
    const uint64_t columns = (uint64_t)a.M * a.batch;
    if (2 * columns < (uint64_t)C::TU * deviceCUs()) return launchIpColsAs<T, P, NF, true>(a, stream);
  }
  return launchIpColsAs<T, P, NF, false>(a, stream);
}

// Most equal factors per launch: as many as 64 to 80 KB of LDS hold at 128 bytes per row.
uint32_t colsInplaceMost(uint32_t P, DType dt) {
  static const uint32_t most[9] = {0, 0, 6, 5, 4, 4, 3, 3, 3};
  return P < 2 || P > 8 ? 0 : most[P];
}
bool colsInplaceFits(uint32_t nf, const uint32_t* p, const uint32_t* q, uint64_t Kin, DType dt) {
  uint64_t K = 1;
  for (uint32_t j = 0; j < nf; j++) {
    if (p[j] != p[0] || q[j] != p[0]) return false;
    K *= p[j];
  }
  return nf >= 2 && nf <= colsInplaceMost(p[0], dt) && K == Kin;
}
bool colsInplaceSupported(const StepArgs& a, DType dt) {
  if (a.batch == 0 || !colsInplaceFits(a.nf, a.p, a.q, a.Kin, dt) || a.Kin != a.Kout) return false;
  if (a.in_ldm != 1 || a.out_ldm != 1 || a.in_ldc != (int64_t)a.M || a.out_ldc != (int64_t)a.M) return false;
  if (a.y && (a.y_ldm != 1 || a.y_ldc != (int64_t)a.M)) return false;
  uint32_t own = 0;
  for (uint32_t j = 0; j < a.nf; j++) {
    if (!(a.f_sq[j] == 1 && a.f_sp[j] == (int64_t)a.q[j]) && !(a.f_sp[j] == 1 && a.f_sq[j] == (int64_t)a.p[j])) return false;
    if (a.batch > 1 && a.f_batch[j] != 0) own++;
  }
  // factors of every entry's own, or none; columns are numbered in 31 bits, offsets inside a tile are
  if (own != 0 && (own != a.nf || a.batch > 65535)) return false;
  if ((uint64_t)a.M * (own ? 1 : a.batch) >= (1ull << 31)) return false;
  const uint64_t widest = std::max({a.in_batch, a.out_batch, a.y ? a.y_batch : 0}), entries = own ? 1 : std::min<uint64_t>(a.batch, 64 / a.M + 2);
  return ((entries - 1) * widest + a.Kin * a.M) * dtypeSize(dt) < (1ull << 31) - 64;
}
hipError_t launchColsInplace(const StepArgs& a, DType dt, hipStream_t stream) {
  if (!colsInplaceSupported(a, dt)) return hipErrorInvalidValue;
#define IP_COLS(P, NF) case P * 16 + NF: return dt == DType::F32 ? launchIpCols<float, P, NF>(a, stream) : launchIpCols<double, P, NF>(a, stream);
  switch (a.p[0] * 16 + a.nf) {
    IP_COLS(2, 2) IP_COLS(2, 3) IP_COLS(2, 4) IP_COLS(2, 5) IP_COLS(2, 6) IP_COLS(3, 2) IP_COLS(3, 3) IP_COLS(3, 4) IP_COLS(3, 5)
    IP_COLS(4, 2) IP_COLS(4, 3) IP_COLS(4, 4) IP_COLS(5, 2) IP_COLS(5, 3) IP_COLS(5, 4) IP_COLS(6, 2) IP_COLS(6, 3)
    IP_COLS(7, 2) IP_COLS(7, 3) IP_COLS(8, 2) IP_COLS(8, 3)
    default: return hipErrorInvalidValue;
  }
#undef IP_COLS
}

hipError_t launchSmallInplace(const StepArgs& a, DType dt, hipStream_t stream) {
  InplaceTile t;
  if (!smallInplaceSupported(a, dt) || !ipTile(a.nf, a.p, a.q, a.Kin, a.M, a.batch, dt, &t)) return hipErrorInvalidValue;
  bool taken;
  if (const hipError_t e = launchIpRowsAny(a, t, dt, stream, &taken); taken || e != hipSuccess) return e;
  return dt == DType::F32 ? launchIpT<float>(a, t, stream) : launchIpT<double>(a, t, stream);
}

}  // namespace fk
