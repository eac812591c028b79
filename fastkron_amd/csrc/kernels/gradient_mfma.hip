// Backward pass of one sliced-multiply step, fp32 or fp64, MKM or KMM layout, any factor shape.
//
// The step computed out[m, q*S + s] = sum_p in[m, s*P + p] F[p, q].  With g = the gradient of `out`, one launch computes
//   gin[m, s*P + p] = sum_q g[m, q*S + s] F[p, q]          (gradient of the step's input)
//   dF[p, q]        = sum_{m,s} in[m, s*P + p] g[m, q*S + s]
// reading `in` and g once from memory.  A row index u runs over all (m, s); it is split as u = o*Tn + t so that both
// layouts have constant strides (MKM: o = m, t = s; KMM: o = s, t = m).
//
// Both products are contractions on V_MFMA_*_16X16X4 without LDS for the operands and without barriers in the loop:
//   dF   A operand lane (k, i) = in[u = 4k+c][p = i], B operand lane (k, j) = g[q = j][u = 4k+c], c = 0..3: the
//        contraction index is permuted so that a lane reads four consecutive u in one 16-byte load where u is the
//        contiguous dimension (g always, `in` in the KMM layout);
//   gin  A operand lane (k, i) = F[p = i][q = 4c+k] from LDS, B operand lane (k, j) = g[q = 4c+k][u = j]: g is read a
//        second time in this order, from the first-level cache.  The rows of F are permuted in fp64 so that a lane ends
//        up with four consecutive p in either type: one 16-byte store (two in fp64) in the MKM layout.
// A wave takes tiles of 16 u; dF stays in its accumulators over all of them, is summed over the four waves of the
// workgroup by a tree in LDS and written as one partial sum per workgroup; kron_grad_reduce_kernel adds the partial sums in a
// fixed order (no atomics: repeated calls give the same bits).
//
// A workgroup handles at most 64x64 of the factor; larger factors run as one launch for dF, one 64x64 block of it per
// grid z, and one for gin, 64 rows of F per grid z with all of Q contracted.
//
// Bound: memory for P, Q <= 32, matrix cores above.  sgemkm 4096 x 32x32^2: 16.7 us a step for 52.6 MB (3.1 TB/s); dgekmm
// 8x8^5 x 16: 7.0 us a step for 12.9 MB, most of it the launch and one tile's round trips.  gin alone falls behind a GEMM
// beyond 128 rows or columns; the PyTorch front end has products of its own there.
// The reference leaves this to PyTorch's matmul (reference pyfastkron/fastkrontorch.py:160-217).
#include <hip/hip_runtime.h>
#include "../problem.h"
#include "gradient.h"
#include "launch.h"

namespace fk {

typedef double gd4 __attribute__((ext_vector_type(4)));
typedef float gf4 __attribute__((ext_vector_type(4)));

template <typename T> struct GMfma;
template <> struct GMfma<double> {
  using V4 = gd4;
  static __device__ __forceinline__ V4 mma(double a, double b, V4 c) { return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0); }
  static __device__ __forceinline__ int row(int r, int hi) { return 4 * r + hi; }
  // which row of F operand row i holds, so that register r of lane group hi is row 4*hi + r of the product
  static __device__ __forceinline__ int perm(int i) { return 4 * (i & 3) + (i >> 2); }
};
template <> struct GMfma<float> {
  using V4 = gf4;
  static __device__ __forceinline__ V4 mma(float a, float b, V4 c) { return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0); }
  static __device__ __forceinline__ int row(int r, int hi) { return 4 * hi + r; }
  static __device__ __forceinline__ int perm(int i) { return i; }
};

constexpr int kGradWaves = 4;
constexpr int kGradThreads = 64 * kGradWaves;

__device__ __forceinline__ uint32_t gradDiv(uint32_t u, const GradStepArgs& a) {
  // exact u / Tn for u < 2^31 (round-up reciprocal)
  return a.tnMagic ? (uint32_t)(((uint64_t)u * a.tnMagic) >> a.tnShift) : u;
}

// ZB: 16-wide blocks of the factor per workgroup in either direction; FULL: P and Q are multiples of 16 * ZB
template <typename T, int ZB, bool DF, bool GA, bool FULL>
__global__ __launch_bounds__(kGradThreads, ZB * ZB * sizeof(T) > 64 ? 1 : (ZB == 4 || sizeof(T) * ZB > 8 ? 2 : 4))
void kron_grad_step_kernel(const GradStepArgs a) {
  using MF = GMfma<T>;
  using V4 = typename MF::V4;
  constexpr int VE = 16 / sizeof(T);                       // elements per 16-byte access
  typedef T VT __attribute__((ext_vector_type(VE)));
  extern __shared__ __align__(16) unsigned char gradLds[];
  T* fs = (T*)gradLds;
  const int tid = threadIdx.x;
  const int l = tid & 63, lo = l & 15, hi = l >> 4;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const uint32_t bt = blockIdx.y;
  const uint32_t P = a.P, Q = a.Q, U = a.U;
  // block of the factor this workgroup works on: (p0, q0) for dF; rows p0 and all q for gin alone
  const uint32_t zq = DF ? blockIdx.z % a.qChunks : 0, zp = DF ? blockIdx.z / a.qChunks : blockIdx.z;
  const uint32_t p0 = zp * (16 * ZB), q0 = zq * (16 * ZB);
  const T* in = (const T*)a.in + (size_t)bt * a.in_batch;
  const T* g = (const T*)a.g + (size_t)bt * a.g_batch;
  const T* F = (const T*)a.f + (size_t)bt * a.f_batch;
  T* gin = GA ? (T*)a.gin + (size_t)bt * a.gin_batch : nullptr;
  const uint32_t nqb = DF ? ZB : (Q + 15) / 16;            // 16-wide blocks of q that gin contracts
  const uint32_t pitch = a.fPitch;                         // LDS elements per row of F (0: F is read from memory)

  if (GA && pitch) {
    // rows p0 .. p0 + 16*ZB of F, zero beyond P and Q; the loads of eight elements in flight (one at a time, 64x64 took
    // 16 round trips to memory, more than the tile of a wave)
    const uint32_t cols = DF ? 16 * ZB : nqb * 16, total = 16 * ZB * cols;
    constexpr int LU = 8;
    // along the contiguous dimension of F
    const bool pFast = a.f_sp == 1;
    for (uint32_t e0 = tid; e0 < total; e0 += LU * kGradThreads) {
      T v[LU];
#pragma unroll
      for (int k = 0; k < LU; k++) {
        const uint32_t e = e0 + k * kGradThreads;
        const uint32_t pl = pFast ? e % (16 * ZB) : e / cols, q = pFast ? e / (16 * ZB) : e - e / cols * cols, p = p0 + pl;
        v[k] = (T)0;
        if (e < total && p < P && q < Q) v[k] = F[(int64_t)p * a.f_sp + (int64_t)q * a.f_sq];
      }
#pragma unroll
      for (int k = 0; k < LU; k++) {
        const uint32_t e = e0 + k * kGradThreads;
        const uint32_t pl = pFast ? e % (16 * ZB) : e / cols, q = pFast ? e / (16 * ZB) : e - e / cols * cols;
        if (e < total) fs[pl * pitch + q] = v[k];
      }
    }
    __syncthreads();
  }
  V4 acc[DF ? ZB : 1][DF ? ZB : 1];
  if (DF) {
#pragma unroll
    for (int i = 0; i < ZB; i++)
#pragma unroll
      for (int j = 0; j < ZB; j++) acc[i][j] = (V4){0, 0, 0, 0};
  }

  // small factors: the second reading of g is requested together with the first
  constexpr bool EARLY = GA && DF && ZB <= 2;
  // element q = qs + hi of a row of g (qs the same for all lanes), clamped to the last one
  const int64_t hiOff = (int64_t)hi * a.g_q;
  auto loadQ = [&](const T* row, uint32_t qs) -> T {
    if (FULL) return (row + hiOff)[(int64_t)qs * a.g_q];
    const uint32_t q = qs + hi;
    return row[(int64_t)(q < Q ? q : Q - 1) * a.g_q];
  };
  // offsets of rows p0 + 16*i + lo of `in` and q0 + 16*i + lo of g
  const int64_t pOff = (int64_t)(p0 + lo) * a.in_p, qOff = (int64_t)(q0 + lo) * a.g_q;
  auto rowP = [&](int i) -> int64_t {
    if (FULL) return pOff + (int64_t)(16 * i) * a.in_p;
    const uint32_t p = p0 + 16 * i + lo;
    return (int64_t)(p < P ? p : P - 1) * a.in_p;
  };
  auto rowQ = [&](int i) -> int64_t {
    if (FULL) return qOff + (int64_t)(16 * i) * a.g_q;
    const uint32_t q = q0 + 16 * i + lo;
    return (int64_t)(q < Q ? q : Q - 1) * a.g_q;
  };
  const uint32_t nWaves = gridDim.x * kGradWaves;
  const uint32_t tiles = (U + 15) / 16;
  for (uint32_t t = blockIdx.x * kGradWaves + w; t < tiles; t += nWaves) {
    const uint32_t u0 = t * 16;
    T gg[EARLY ? 4 * ZB : 1];
    int64_t ginOff = 0;
    const T* gu = nullptr;
    if (GA) {
      const uint32_t u = u0 + lo < U ? u0 + lo : U - 1;
      const uint32_t o = gradDiv(u, a), tt = u - o * a.Tn;
      ginOff = (int64_t)o * a.in_o + (int64_t)tt * a.in_t;
      gu = g + (int64_t)o * a.g_o + (int64_t)tt * a.g_t;
      if (EARLY) {
#pragma unroll
        for (int c = 0; c < 4 * ZB; c++) gg[c] = loadQ(gu, 4 * c);
      }
    }
    if (DF) {
      T av[ZB][4], gv[ZB][4];
      const uint32_t ub = u0 + 4 * hi;
      if (a.vecIn || a.vecG) {
        // Tn is a multiple of four: the four u of a lane are neighbours in one run of t, and all below U or none
        const bool ok = ub < U;
        const uint32_t u = ok ? ub : 0;
        const uint32_t o = gradDiv(u, a), tt = u - o * a.Tn;
        const T* ip = in + (int64_t)o * a.in_o + (int64_t)tt * a.in_t;
        const T* gp = g + (int64_t)o * a.g_o + (int64_t)tt * a.g_t;
#pragma unroll
        for (int i = 0; i < ZB; i++) {
          const int64_t po = rowP(i), qo = rowQ(i);
          if (a.vecIn) {
#pragma unroll
            for (int v = 0; v < 4 / VE; v++) {
              const VT x = *(const VT*)(ip + po + v * VE);
#pragma unroll
              for (int e = 0; e < VE; e++) av[i][v * VE + e] = x[e];
            }
          } else {
#pragma unroll
            for (int c = 0; c < 4; c++) av[i][c] = ip[(int64_t)c * a.in_t + po];
          }
          if (a.vecG) {
#pragma unroll
            for (int v = 0; v < 4 / VE; v++) {
              const VT x = *(const VT*)(gp + qo + v * VE);
#pragma unroll
              for (int e = 0; e < VE; e++) gv[i][v * VE + e] = x[e];
            }
          } else {
#pragma unroll
            for (int c = 0; c < 4; c++) gv[i][c] = gp[(int64_t)c * a.g_t + qo];
          }
        }
        if (!ok) {
#pragma unroll
          for (int i = 0; i < ZB; i++)
#pragma unroll
            for (int c = 0; c < 4; c++) { av[i][c] = (T)0; gv[i][c] = (T)0; }
        }
      } else {
#pragma unroll
        for (int c = 0; c < 4; c++) {
          const bool ok = ub + c < U;
          const uint32_t u = ok ? ub + c : 0;
          const uint32_t o = gradDiv(u, a), tt = u - o * a.Tn;
          const T* ip = in + (int64_t)o * a.in_o + (int64_t)tt * a.in_t;
          const T* gp = g + (int64_t)o * a.g_o + (int64_t)tt * a.g_t;
#pragma unroll
          for (int i = 0; i < ZB; i++) {
            const T x = ip[rowP(i)], y = gp[rowQ(i)];
            av[i][c] = ok ? x : (T)0;
            gv[i][c] = ok ? y : (T)0;
          }
        }
      }
#pragma unroll
      for (int c = 0; c < 4; c++)
#pragma unroll
        for (int i = 0; i < ZB; i++)
#pragma unroll
          for (int j = 0; j < ZB; j++) acc[i][j] = MF::mma(av[i][c], gv[j][c], acc[i][j]);
    }
    if (GA) {
      V4 ga[ZB];
#pragma unroll
      for (int i = 0; i < ZB; i++) ga[i] = (V4){0, 0, 0, 0};
      // (a 64x64 block of F does not fit the registers beside the sums: its reads stay in the loop)
      int fLane = MF::perm(lo) * (int)pitch + hi;
      if (ZB == 4) asm volatile("" : "+v"(fLane));
      auto contract = [&](uint32_t qb, const T (&x)[4]) {
#pragma unroll
        for (int c = 0; c < 4; c++) {
          const uint32_t q = 16 * qb + 4 * c + hi;
          const T xv = FULL || q < Q ? x[c] : (T)0;
#pragma unroll
          for (int i = 0; i < ZB; i++) {
            T f;
            if (DF || pitch) f = fs[fLane + 16 * i * pitch + 16 * qb + 4 * c];
            else {
              const uint32_t pl = 16 * i + MF::perm(lo);
              const uint32_t p = p0 + pl < P ? p0 + pl : P - 1;
              // (as in LDS, zero beyond Q: an infinity in the last column would count as 0 * inf)
              const T v = F[(int64_t)p * a.f_sp + (int64_t)(q < Q ? q : Q - 1) * a.f_sq];
              f = FULL || q < Q ? v : (T)0;
            }
            ga[i] = MF::mma(f, xv, ga[i]);
          }
        }
      };
      if (DF) {
#pragma unroll
        for (int qb = 0; qb < ZB; qb++) {
          T x[4];
#pragma unroll
          for (int c = 0; c < 4; c++) x[c] = EARLY ? gg[EARLY ? 4 * qb + c : 0] : loadQ(gu, 16 * qb + 4 * c);
          if (FULL || 16u * qb < Q) contract(qb, x);
        }
      } else {
        for (uint32_t qb = 0; qb < nqb; qb++) {
          T x[4];
#pragma unroll
          for (int c = 0; c < 4; c++) x[c] = loadQ(gu, 16 * qb + 4 * c);
          contract(qb, x);
        }
      }
      if (u0 + lo < U) {
        T* op = gin + ginOff;
#pragma unroll
        for (int i = 0; i < ZB; i++) {
          const uint32_t p = p0 + 16 * i + 4 * hi;
          if (a.vecOut) {                                  // P a multiple of four, p contiguous
            if (FULL || p < P) {
#pragma unroll
              for (int v = 0; v < 4 / VE; v++) {
                VT x;
#pragma unroll
                for (int e = 0; e < VE; e++) x[e] = ga[i][v * VE + e];
                *(VT*)(op + p + v * VE) = x;
              }
            }
          } else {
#pragma unroll
            for (int r = 0; r < 4; r++)
              if (FULL || p + r < P) op[(int64_t)(p + r) * a.in_p] = ga[i][r];
          }
        }
      }
    }
  }

  if (DF) {
    // the four waves' sums as a tree in LDS: (0 + 2) + (1 + 3), a lane's values side by side for all lanes
    constexpr int N = 16 * ZB;
    static_assert(kGradWaves == 4, "two levels");
    auto slot = [&](int half, int i, int j, int r) { return fs + half * (N * N) + ((i * ZB + j) * 4 + r) * 64 + l; };
    __syncthreads();                                       // everyone is done with the factor in LDS
    if (w >= 2) {
#pragma unroll
      for (int i = 0; i < ZB; i++)
#pragma unroll
        for (int j = 0; j < ZB; j++)
#pragma unroll
          for (int r = 0; r < 4; r++) *slot(w - 2, i, j, r) = acc[i][j][r];
    }
    __syncthreads();
    if (w < 2) {
#pragma unroll
      for (int i = 0; i < ZB; i++)
#pragma unroll
        for (int j = 0; j < ZB; j++)
#pragma unroll
          for (int r = 0; r < 4; r++) acc[i][j][r] += *slot(w, i, j, r);
    }
    __syncthreads();
    if (w == 1) {
#pragma unroll
      for (int i = 0; i < ZB; i++)
#pragma unroll
        for (int j = 0; j < ZB; j++)
#pragma unroll
          for (int r = 0; r < 4; r++) *slot(0, i, j, r) = acc[i][j][r];
    }
    __syncthreads();
    if (w == 0) {
      // (the second half holds the block row by row for the store)
#pragma unroll
      for (int i = 0; i < ZB; i++)
#pragma unroll
        for (int j = 0; j < ZB; j++)
#pragma unroll
          for (int r = 0; r < 4; r++)
            fs[N * N + (16 * i + MF::row(r, hi)) * N + 16 * j + lo] = acc[i][j][r] + *slot(0, i, j, r);
    }
    __syncthreads();
    T* part = (T*)a.partial + ((size_t)bt * a.partStride + a.partFirst + blockIdx.x) * ((size_t)P * Q);
    for (uint32_t e = tid; e < N * N; e += kGradThreads) {
      const uint32_t pl = a.partSq == 1 ? e / N : e % N, ql = a.partSq == 1 ? e % N : e / N, p = p0 + pl, q = q0 + ql;
      if (p < P && q < Q) part[(size_t)p * a.partSp + (size_t)q * a.partSq] = fs[N * N + pl * N + ql];
    }
  }
}

// dF[p, q] = sum over the partial sums, all factors (grid y) and batch entries (grid z) of a backward pass in one launch.
// A workgroup takes 32 entries and splits the partial sums eight ways.
template <typename T>
__global__ __launch_bounds__(256) void kron_grad_reduce_kernel(const GradReduceArgs a) {
  const GradReduce r = a.r[blockIdx.y];
  __shared__ T s[8][33];
  const int e = threadIdx.x & 31, k = threadIdx.x >> 5;
  const uint32_t n = r.P * r.Q;
  for (uint32_t base = blockIdx.x * 32; base < n; base += gridDim.x * 32) {
    const uint32_t idx = base + e;
    const T* src = (const T*)r.partial + (size_t)blockIdx.z * r.count * n;
    T v0 = (T)0, v1 = (T)0, v2 = (T)0, v3 = (T)0;
    if (idx < n) {
      uint32_t i = k;
      for (; i + 24 < r.count; i += 32) {
        v0 += src[(size_t)i * n + idx];
        v1 += src[(size_t)(i + 8) * n + idx];
        v2 += src[(size_t)(i + 16) * n + idx];
        v3 += src[(size_t)(i + 24) * n + idx];
      }
      for (; i < r.count; i += 8) v0 += src[(size_t)i * n + idx];
    }
    s[k][e] = (v0 + v1) + (v2 + v3);
    __syncthreads();
    if (k == 0 && idx < n) {
      T v = s[0][e];
#pragma unroll
      for (int j = 1; j < 8; j++) v += s[j][e];
      const uint32_t p = idx / r.Q, q = idx - p * r.Q;
      ((T*)r.out)[(size_t)blockIdx.z * n + (size_t)p * r.osp + (size_t)q * r.osq] = v;
    }
    __syncthreads();
  }
}

template <typename T, int ZB, bool DF, bool GA, bool FULL>
static hipError_t launchGradF(const GradStepArgs& a, uint32_t gridX, uint32_t gridZ, size_t lds, hipStream_t stream) {
  static PerDeviceOnce attrOnce;
  const int devIdx = launchDeviceIndex();
  if (lds > 65536 && !attrOnce.done(devIdx)) {
    hipError_t e = hipFuncSetAttribute((const void*)kron_grad_step_kernel<T, ZB, DF, GA, FULL>, hipFuncAttributeMaxDynamicSharedMemorySize,
                                       (int)kGradLdsMax);
    if (e != hipSuccess) return e;
    attrOnce.mark(devIdx);
  }
  hipLaunchKernelGGL((kron_grad_step_kernel<T, ZB, DF, GA, FULL>), dim3(gridX, a.batch, gridZ), dim3(kGradThreads), lds, stream, a);
  return hipGetLastError();
}

template <typename T, int ZB, bool DF, bool GA>
static hipError_t launchGradT(const GradStepArgs& a, uint32_t gridX, uint32_t gridZ, size_t lds, hipStream_t stream) {
  const bool full = a.P % (16 * ZB) == 0 && a.Q % (16 * ZB) == 0;
  return full ? launchGradF<T, ZB, DF, GA, true>(a, gridX, gridZ, lds, stream) : launchGradF<T, ZB, DF, GA, false>(a, gridX, gridZ, lds, stream);
}

uint32_t gradWorkgroups(uint32_t P, uint32_t Q, uint64_t U, uint32_t batch) {
  const uint64_t tiles = (U + 15) / 16, need = (tiles + kGradWaves - 1) / kGradWaves;
  const uint32_t big = P > Q ? P : Q;
  const uint64_t share = (uint64_t)batch * ((P + 63) / 64) * ((Q + 63) / 64);
  uint64_t cap = 1;
  if (big <= 32) {
    if (share < 512) cap = 512 / share;
  } else {
    // The number for which the last 256 CUs' worth of workgroups is fullest, the smallest of equal ones, within four times 256.
    // Rounded up from 256 / blocks, 3x3 blocks had 261 workgroups, which took as long as 512 (forward pass and factor gradient, us:
    // sgekmm 192x192 x 83333 484 -> 353, 96x192 x 83333 271 -> 191, 640x640 x 6250 367 -> 279).
    for (uint64_t c = 1; c * share <= 1024; c++)
      if ((c * share + 255) / 256 * cap < (cap * share + 255) / 256 * c) cap = c;
  }
  return (uint32_t)(need < cap ? need : cap);
}

template <typename T>
static hipError_t launchGradStepT(GradStepArgs a, hipStream_t stream) {
  const uint32_t big = a.P > a.Q ? a.P : a.Q;
  const int zb = big <= 16 ? 1 : big <= 32 ? 2 : 4;
  const uint32_t pChunks = (a.P + 16 * zb - 1) / (16 * zb), qBlocks = (a.Q + 15) / 16;
  a.qChunks = (a.Q + 16 * zb - 1) / (16 * zb);
  const size_t red = (size_t)2 * 256 * zb * zb * sizeof(T);           // two halves of the tree
  auto run = [&](auto df, auto ga, uint32_t gridX, uint32_t gridZ) -> hipError_t {
    constexpr bool D = decltype(df)::value, G = decltype(ga)::value;
    const uint32_t cols = D ? 16 * zb : 16 * qBlocks;
    size_t lds = G ? (size_t)16 * zb * (cols + 4) * sizeof(T) : 0;
    a.fPitch = cols + 4;
    if (lds > kGradLdsMax) { lds = 0; a.fPitch = 0; }
    if (D && red > lds) lds = red;
    if (zb == 1) return launchGradT<T, 1, D, G>(a, gridX, gridZ, lds, stream);
    if (zb == 2) return launchGradT<T, 2, D, G>(a, gridX, gridZ, lds, stream);
    return launchGradT<T, 4, D, G>(a, gridX, gridZ, lds, stream);
  };
  using Yes = std::integral_constant<bool, true>;
  using No = std::integral_constant<bool, false>;
  const bool one = pChunks == 1 && a.qChunks == 1;
  if (a.partial && a.gin && one) return run(Yes{}, Yes{}, a.gridX, 1);
  hipError_t e = hipSuccess;
  if (a.partial) e = run(Yes{}, No{}, a.gridX, pChunks * a.qChunks);
  if (e == hipSuccess && a.gin) {
    const uint64_t need = ((a.U + 15) / 16 + kGradWaves - 1) / kGradWaves;
    uint64_t cap = 1024 / ((uint64_t)a.batch * pChunks);
    if (cap < 1) cap = 1;
    e = run(No{}, Yes{}, (uint32_t)(need < cap ? need : cap), pChunks);
  }
  return e;
}

hipError_t launchGradStep(const GradStepArgs& a, DType dt, hipStream_t stream) {
  if (a.U == 0 || a.U >= (1u << 31) || a.batch == 0 || a.batch > 65535 || a.P == 0 || a.Q == 0 || (!a.partial && !a.gin))
    return hipErrorInvalidValue;
  return dt == DType::F32 ? launchGradStepT<float>(a, stream) : launchGradStepT<double>(a, stream);
}

hipError_t launchGradReduce(const GradReduceArgs& a, uint32_t batch, DType dt, hipStream_t stream) {
  if (a.count == 0) return hipSuccess;
  uint32_t widest = 0;
  for (uint32_t i = 0; i < a.count; i++) widest = a.r[i].P * a.r[i].Q > widest ? a.r[i].P * a.r[i].Q : widest;
  uint32_t gx = (widest + 31) / 32;
  if (gx > 4096) gx = 4096;
  const dim3 grid(gx, a.count, batch);
  if (dt == DType::F32) hipLaunchKernelGGL(kron_grad_reduce_kernel<float>, grid, dim3(256), 0, stream, a);
  else                  hipLaunchKernelGGL(kron_grad_reduce_kernel<double>, grid, dim3(256), 0, stream, a);
  return hipGetLastError();
}

}  // namespace fk
