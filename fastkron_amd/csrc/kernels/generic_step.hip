// Fallback kernel: one sliced-multiply step for any P, Q, strides and operand transposes.
//
//   out[m, q*S + s] = sum_p in[m, s*P + p] * F[p, q],   S = Kin / P
//
// (step semantics as in reference tests/testBase.h:256-283; it plays the role of the reference's
// low-optimisation-level kernels, src/kernels/kernel_opt.h:42-84.)  Every thread owns one (row, slice)
// pair and TQ output columns; the factor chunk is staged in LDS and read as a broadcast.  Lanes run
// along the rows when rows are the contiguous dimension of the input (KMM layout) and along slices
// otherwise, so that stores are coalesced in both layouts.
#include <hip/hip_runtime.h>
#include "../problem.h"
#include "launch.h"

namespace fk {

constexpr int kGenThreads = 256;
constexpr int kGenTP = 32;

template <typename T, int TQ, bool LANES_M, bool AHEAD>
__global__ __launch_bounds__(kGenThreads) void kron_step_generic(const KernelArgs a, const uint32_t qTiles, const OuterStrides outer) {
  __shared__ T fs[kGenTP][TQ];
  const uint32_t P = a.p[0], Q = a.q[0];
  const uint64_t S = a.Kin / P;
  const uint64_t tile = blockIdx.x / qTiles;
  const uint32_t q0 = (blockIdx.x % qTiles) * TQ;
  const uint32_t b = blockIdx.z;
  const T* in = (const T*)a.in + (size_t)b * a.in_batch + (size_t)blockIdx.y * outer.in;
  T* out = (T*)a.out + (size_t)b * a.out_batch + (size_t)blockIdx.y * outer.out;
  const T* y = a.y ? (const T*)a.y + (size_t)b * a.y_batch + (size_t)blockIdx.y * outer.y : nullptr;
  const T* F = (const T*)a.f[0] + (size_t)b * a.f_batch[0];

  const uint64_t g = tile * kGenThreads + threadIdx.x;
  const bool active = g < (uint64_t)a.M * S;
  uint64_t m, s;
  if (LANES_M) { m = g % a.M; s = g / a.M; } else { s = g % S; m = g / S; }

  T acc[TQ];
#pragma unroll
  for (int i = 0; i < TQ; i++) acc[i] = T(0);

  const T* xrow = in + (int64_t)m * a.in_ldm + (int64_t)(s * P) * a.in_ldc;
  auto stage = [&](uint32_t p0) {
    for (uint32_t idx = threadIdx.x; idx < kGenTP * TQ; idx += kGenThreads) {
      const uint32_t pp = p0 + idx / TQ, qq = q0 + idx % TQ;
      fs[idx / TQ][idx % TQ] = (pp < P && qq < Q) ? F[(int64_t)pp * a.f_sp[0] + (int64_t)qq * a.f_sq[0]] : T(0);
    }
    __syncthreads();
  };
  if constexpr (AHEAD) {
    // eight elements of X in registers ahead of their products, the first eight ahead of the factor's
    constexpr int LU = 8;
    T x[LU];
    auto loadX = [&](uint32_t p) {
#pragma unroll
      for (int u = 0; u < LU; u++) {
        x[u] = T(0);
        if (p + u < P && active) x[u] = xrow[(int64_t)(p + u) * a.in_ldc];
      }
    };
    loadX(0);
    for (uint32_t p0 = 0; p0 < P; p0 += kGenTP) {
      if (p0) __syncthreads();
      stage(p0);
      const uint32_t pn = (P - p0 < (uint32_t)kGenTP) ? P - p0 : kGenTP;
      for (uint32_t pp = 0; pp < pn; pp += LU) {
        T xc[LU];
#pragma unroll
        for (int u = 0; u < LU; u++) xc[u] = x[u];
        if (p0 + pp + LU < P) loadX(p0 + pp + LU);
#pragma unroll
        for (int u = 0; u < LU; u++) {
          if (pp + u >= pn) break;
#pragma unroll
          for (int i = 0; i < TQ; i++) acc[i] += xc[u] * fs[pp + u][i];
        }
      }
    }
  } else {
    for (uint32_t p0 = 0; p0 < P; p0 += kGenTP) {
      __syncthreads();
      stage(p0);
      if (active) {
        const uint32_t pn = (P - p0 < (uint32_t)kGenTP) ? P - p0 : kGenTP;
        for (uint32_t pp = 0; pp < pn; pp++) {
          const T x = xrow[(int64_t)(p0 + pp) * a.in_ldc];
#pragma unroll
          for (int i = 0; i < TQ; i++) acc[i] += x * fs[pp][i];
        }
      }
    }
  }
  if (!active) return;
  const T alpha = (T)a.alpha, beta = (T)a.beta;
#pragma unroll
  for (int i = 0; i < TQ; i++) {
    const uint32_t q = q0 + i;
    if (q >= Q) break;
    const uint64_t col = (uint64_t)q * S + s;
    T v = acc[i];
    if (a.epilogue) {
      v = alpha * v;
      if (y) v += beta * y[(int64_t)m * a.y_ldm + (int64_t)col * a.y_ldc];
    }
    out[(int64_t)m * a.out_ldm + (int64_t)col * a.out_ldc] = v;
  }
}

template <typename T, bool LANES_M>
static hipError_t launchGenericT(const StepArgs& a, hipStream_t stream) {
  const uint32_t Q = a.q[0];
  const uint64_t S = a.Kin / a.p[0];
  const uint64_t tiles = ((uint64_t)a.M * S + kGenThreads - 1) / kGenThreads;
  int tq = 1;
  while (tq < 16 && (uint32_t)tq < Q) tq *= 2;
  // few workgroups: fewer output columns per thread and more threads, which read X through the caches
  while (tq > 4 && tiles * ((Q + tq - 1) / tq) * a.batch < 128) tq /= 2;
  const uint32_t qTiles = (Q + tq - 1) / tq;
  if (tiles * qTiles >= (1ull << 31) || a.batch > 65535) return hipErrorInvalidValue;
  dim3 grid((uint32_t)(tiles * qTiles), outerEntries(a), innerEntries(a)), block(kGenThreads);
  // Loads ahead of the products, up to four workgroups per CU: for short rows, where the first eight leave before the factor
  // is staged (sgekmm 7^5 x 100 37.0 -> 34.7 us, 17^3 x 200 27.5 -> 24.8, 3^8 x 50 34.3 -> 30.0), and in the KMM layout where
  // a load takes long: few columns and with them many short pieces (21^3 x 25, batch of 5, 29.0 -> 24.7), or an X of more
  // than an XCD's L2 has left (dgekmm 129^2 x 60 76 -> 61, 257x40 x 30000 70 -> 55, 300^2 x 7 140 -> 101; with few output
  // columns per thread, whose products hide little, beyond 32 MB, 512x1 x 30000 57 -> 47).  Elsewhere rows of more than 32
  // elements run into the staging of the next 32 with nothing gained and the plain loop is ahead (1000x3, one row, 42 us
  // against 84, 2048x2048, 7 rows, 212 / 316, dgemkm 40x3^3 x 30 20.8 / 24.3), and so it is on full devices, where the waves
  // of a CU hide each other's round trips (27^3 x 21, batch of 10, 1200 workgroups, 40.5 / 42.3).
  const uint32_t P = a.p[0];
  const uint64_t wgs = tiles * qTiles * a.batch, xBytes = (uint64_t)a.M * a.Kin * a.batch * sizeof(T);
  const bool ahead = wgs < 1024 && (P <= 20 || (LANES_M && (P <= 32 ? a.M < 128 && S > 1 : xBytes >= (tq >= 8 ? 2400000u : 32000000u))));
#define GEN_LAUNCH(TQ) \
  if (ahead) hipLaunchKernelGGL((kron_step_generic<T, TQ, LANES_M, true>), grid, block, 0, stream, a, qTiles, a.outer); \
  else       hipLaunchKernelGGL((kron_step_generic<T, TQ, LANES_M, false>), grid, block, 0, stream, a, qTiles, a.outer);
  switch (tq) {
    case 1:  GEN_LAUNCH(1) break;
    case 2:  GEN_LAUNCH(2) break;
    case 4:  GEN_LAUNCH(4) break;
    case 8:  GEN_LAUNCH(8) break;
    default: GEN_LAUNCH(16) break;
  }
#undef GEN_LAUNCH
  return hipGetLastError();
}

hipError_t launchGenericStep(const StepArgs& a, DType dt, hipStream_t stream) {
  if (a.nf != 1 || a.M == 0 || a.batch == 0 || a.Kin == 0) return hipErrorInvalidValue;
  const bool lanesM = (a.in_ldm == 1 && a.M > 1);
  if (dt == DType::F32)
    return lanesM ? launchGenericT<float, true>(a, stream) : launchGenericT<float, false>(a, stream);
  return lanesM ? launchGenericT<double, true>(a, stream) : launchGenericT<double, false>(a, stream);
}

}  // namespace fk
