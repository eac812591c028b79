// Two factors of any sizes up to 64 (P1 x Q1 and P2 x Q2, fp32 or fp64) on rows of exactly P1*P2 columns, MKM layout, in one
// launch on the matrix cores (V_MFMA_F32_16X16X4_F32 / V_MFMA_F64_16X16X4_F64): 31x63, 50x50, 24x48, 12x20 ... and the two
// trailing factors of longer chains on contiguous blocks.
//
//   T[p1][q2] = sum_p2 X[p1][p2] F2[p2][q2],    Z[q1][q2] = sum_p1 F1[p1][q1] T[p1][q2]
//
// A wave owns 16 neighbouring columns q2 of a row's result.  Its column block of F2 and all of F1 stay in registers as matrix
// operands (zero beyond the real sizes; F1 in LDS for inputs of more than 32 rows in fp64), and the accumulators of the first product are
// the B operand of the second one, whose contraction index is permuted to match (as in pair_mfma.hip): T never leaves the
// registers.  X arrives as whole 16-byte pieces whatever its alignment, the next tile's on their way while this one is
// multiplied, and goes through LDS to the waves of a row; elements beyond P2 and rows beyond P1 are selected to zero as they
// are read, and the rows beyond P1 of the first product once more (padding with zeros alone would make NaN of an infinity in X
// or F2).  Results go out by quarter waves of 16 consecutive
// elements through a descriptor of the row's result, which drops rows beyond Q1.
//
// Bound: memory for large row counts, for few rows one chain of load, products and store per workgroup.
#include <hip/hip_runtime.h>
#include <algorithm>
#include "../problem.h"
#include "launch.h"

namespace fk {

constexpr uint32_t kPaMax = 64;
constexpr uint32_t kPaThreads = 256;

struct PairAnyTile {
  uint32_t P1, P2, Q1, Q2;
  uint32_t waves, items;            // waves per row (a power of two), rows per workgroup at a time
  uint32_t tiles;
  uint32_t pitchedMagic;            // floor(piece / (P2 / VE)) = mulhi(piece, magic); 0: rows are no whole pieces
};

typedef double Pa64 __attribute__((ext_vector_type(4)));
typedef float Pa32 __attribute__((ext_vector_type(4)));
// row(r, hi): row, within a 16x16 accumulator, of register r in lanes 16*hi ..; rowLane(hi) + rowReg(r)
template <typename T> struct PaMfma;
template <> struct PaMfma<double> {
  using Acc = Pa64;
  static __device__ __forceinline__ Acc mma(double a, double b, Acc c) { return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0); }
  static __device__ __forceinline__ int rowLane(int hi) { return hi; }
  static constexpr int rowReg(int r) { return 4 * r; }
};
template <> struct PaMfma<float> {
  using Acc = Pa32;
  static __device__ __forceinline__ Acc mma(float a, float b, Acc c) { return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0); }
  static __device__ __forceinline__ int rowLane(int hi) { return 4 * hi; }
  static constexpr int rowReg(int r) { return r; }
};

constexpr uint32_t kPaNowhere = 0x7ffffff0u;         // an offset outside every descriptor here

// Rows per workgroup at a time, at most: four waves on 32-wide inputs, two rows of 64-wide ones.
constexpr uint32_t paItems(int PB) { return PB == 2 ? 4 : 2; }

// PB, QB: 16-wide blocks of an input / output digit (2: up to 32, 4: up to 64)
template <typename T, int PB, int QB, bool HAS_Y>
__global__ __launch_bounds__(kPaThreads, 2) void kron_pair_any_kernel(const KernelArgs a, const PairAnyTile t, const OuterStrides outer) {
  using MF = PaMfma<T>;
  using Acc = typename MF::Acc;
  constexpr uint32_t ES = sizeof(T), VE = 16 / ES;
  typedef T VT __attribute__((ext_vector_type(VE)));
  constexpr int PC = PB * 4;                                       // products of the first contraction
  constexpr bool kF1Lds = ES == 8 && PB == 4;
  constexpr int LV = (int)((paItems(PB) * PB * PB * 256 / VE + 1 + kPaThreads - 1) / kPaThreads);
  extern __shared__ __align__(16) unsigned char paLds[];
  const uint32_t tid = threadIdx.x, b = blockIdx.y;
  const int l = tid & 63, lo = l & 15, hi = l >> 4, w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const uint32_t slot = (uint32_t)w / t.waves, jb = (uint32_t)w % t.waves;
  const uint32_t rowIn = t.P1 * t.P2, rowOut = t.Q1 * t.Q2, pc2 = (t.P2 + 3) / 4;
  const bool columns = 16 * jb < t.Q2;
  const T alpha = a.epilogue ? (T)a.alpha : T(1), beta = (T)a.beta;
  VT* pieces = (VT*)paLds;
  T* f1Lds = (T*)paLds;                                             // (behind the tile: see below)

  const T* const inB = (const T*)a.in + (size_t)b * a.in_batch + (size_t)blockIdx.z * outer.in;
  T* const outB = (T*)a.out + (size_t)b * a.out_batch + (size_t)blockIdx.z * outer.out;
  T* const yB = HAS_Y ? (T*)a.y + (size_t)b * a.y_batch + (size_t)blockIdx.z * outer.y : nullptr;
  struct Tile { const T* src; uint32_t n, E, shift, last; };
  auto tileAt = [&](uint32_t i) {
    Tile r;
    const uint32_t m0 = i * t.items;
    r.n = a.M - m0 < t.items ? a.M - m0 : t.items;
    r.E = r.n * rowIn;
    r.src = inB + (size_t)m0 * rowIn;
    r.shift = (uint32_t)((uintptr_t)r.src / ES) & (VE - 1);
    r.last = (r.shift + r.E) / VE;
    return r;
  };
  // (the element, before the first or behind the last 16-byte piece inside the tile, that thread tid takes)
  auto edgeOf = [&](const Tile& r, uint32_t* e) {
    const uint32_t behind = r.last * VE > r.shift ? r.last * VE - r.shift : 0;
    const uint32_t before = r.shift == 0 ? 0 : VE - r.shift < r.E ? VE - r.shift : r.E;
    if (tid < VE) { *e = tid; return tid < before; }
    *e = behind + tid - VE;
    return tid < 2 * VE && *e < r.E && *e >= before;
  };
  VT v[LV];
  T edge = T(0);
  auto fetch = [&](const Tile& r) {
    const auto from = streamTarget((void*)(r.src - r.shift), r.last * 16);
    uint32_t e;
    if (edgeOf(r, &e)) edge = r.src[e];
#pragma unroll
    for (int k = 0; k < LV; k++)
      if (k * kPaThreads < r.last)
        v[k] = __builtin_bit_cast(VT, __builtin_amdgcn_raw_buffer_load_b128(from, (int)(k == 0 && tid == 0 && r.shift ? kPaNowhere : tid * 16),
                                                                           k * kPaThreads * 16, 0));
  };
  uint32_t i = blockIdx.x;
  Tile r = tileAt(i);
  fetch(r);

  // factor operands; the first product takes p2 = pc2*hi + c in step c
  T f2[PC], f1[kF1Lds ? 1 : QB][kF1Lds ? 1 : PB][4];
  {
    const auto F2 = streamTarget((T*)a.f[0] + (size_t)b * a.f_batch[0], t.P2 * t.Q2 * ES);
    const auto F1 = streamTarget((T*)a.f[1] + (size_t)b * a.f_batch[1], t.P1 * t.Q1 * ES);
    const uint32_t q2 = 16 * jb + lo;
#pragma unroll
    for (int c = 0; c < PC; c++) {
      const uint32_t p = pc2 * hi + c;
      const bool in = (uint32_t)c < pc2 && p < t.P2 && q2 < t.Q2;
      f2[c] = bufferLoad<T>(F2, in ? (uint32_t)(p * a.f_sp[0] + q2 * a.f_sq[0]) * ES : kPaNowhere, 0);
    }
    if constexpr (kF1Lds) {
      f1Lds = (T*)(paLds + t.items * t.P1 * (t.P2 + VE) * ES + 64);
      for (uint32_t k = tid; k < 64 * 64; k += kPaThreads) {
        const uint32_t p = k / 64, q = k % 64;
        f1Lds[k] = bufferLoad<T>(F1, p < t.P1 && q < t.Q1 ? (uint32_t)(p * a.f_sp[1] + q * a.f_sq[1]) * ES : kPaNowhere, 0);
      }
    } else {
#pragma unroll
      for (int u = 0; u < QB; u++)
#pragma unroll
        for (int g = 0; g < PB; g++)
#pragma unroll
          for (int k = 0; k < 4; k++) {
            const uint32_t p = 16 * g + MF::rowLane(hi) + MF::rowReg(k), q = 16 * u + lo;
            f1[u][g][k] = bufferLoad<T>(F1, p < t.P1 && q < t.Q1 ? (uint32_t)(p * a.f_sp[1] + q * a.f_sq[1]) * ES : kPaNowhere, 0);
          }
    }
  }

  for (;;) {
    // rows that are whole pieces get a pitch of one more, which spreads a column over the LDS banks
    const bool pitched = t.pitchedMagic != 0 && r.shift == 0;
    const uint32_t pitch = pitched ? t.P2 + VE : t.P2, shift = r.shift;
#pragma unroll
    for (int k = 0; k < LV; k++) {
      const uint32_t c = tid + k * kPaThreads;
      if (c < r.last && (c > 0 || shift == 0)) pieces[pitched ? c + __umulhi(c, t.pitchedMagic) : c] = v[k];
    }
    uint32_t e;
    if (edgeOf(r, &e)) ((T*)paLds)[shift + e] = edge;
    __syncthreads();

    const uint32_t row = i * t.items + slot;
    const bool work = slot < r.n && columns, more = i + gridDim.x < t.tiles;
    if (more) {
      i += gridDim.x;
      r = tileAt(i);
      fetch(r);
    }
    Acc d1[PB];
    if (work) {
      const T* x[PB];
      int limit[PB];                                              // real elements of this lane's run of the row
      const int run = (int)(t.P2 - pc2 * hi) < (int)pc2 ? (int)(t.P2 - pc2 * hi) : (int)pc2;
#pragma unroll
      for (int g = 0; g < PB; g++) {
        const bool in = 16 * g + lo < (int)t.P1;
        x[g] = (const T*)paLds + shift + (slot * t.P1 + (in ? 16 * g + lo : 0)) * pitch + (run > 0 ? pc2 * hi : 0);
        limit[g] = in ? run : 0;
        d1[g] = (Acc){0, 0, 0, 0};
      }
#pragma unroll
      for (int cg = 0; cg < PC / 4; cg++)
        if (4 * cg < (int)pc2) {
#pragma unroll
          for (int g = 0; g < PB; g++)
            if (g == 0 || 16 * g < (int)t.P1) {
              T xv[4];
#pragma unroll
              for (int c = 0; c < 4; c++) xv[c] = x[g][4 * cg + c];
#pragma unroll
              for (int c = 0; c < 4; c++) d1[g] = MF::mma(4 * cg + c < limit[g] ? xv[c] : T(0), f2[4 * cg + c], d1[g]);
            }
        }
      // rows beyond P1 are zero times F2, NaN where that is infinite: they are zero in the second product as well
      // (1003 rows of 31x63^2 10.1 -> 10.4 us; only where a factor is not finite, or without the condition: the same)
#pragma unroll
      for (int g = 0; g < PB; g++)
        if (16 * g < (int)t.P1 && 16 * g + 16 > (int)t.P1) {
#pragma unroll
          for (int k = 0; k < 4; k++)
            if (16 * g + MF::rowLane(hi) + MF::rowReg(k) >= (int)t.P1) d1[g][k] = T(0);
        }
    }
    __syncthreads();                                              // the tile has been read
    if (work) {
      const auto out = streamTarget(outB + (size_t)row * rowOut, rowOut * ES);
      const auto y = HAS_Y ? streamTarget(yB + (size_t)row * rowOut, rowOut * ES) : out;
      const uint32_t q2 = 16 * jb + lo, lane = q2 < t.Q2 ? (MF::rowLane(hi) * t.Q2 + q2) * ES : kPaNowhere;
#pragma unroll
      for (int u = 0; u < QB; u++)
        if (u == 0 || 16 * u < (int)t.Q1) {
          Acc z = {0, 0, 0, 0};
          T yv[4];
#pragma unroll
          for (int k = 0; k < 4; k++) yv[k] = HAS_Y ? bufferLoad<T>(y, lane, (16 * u + MF::rowReg(k)) * t.Q2 * ES) : T(0);
#pragma unroll
          for (int g = 0; g < PB; g++)
            if (g == 0 || 16 * g < (int)t.P1) {
#pragma unroll
              for (int k = 0; k < 4; k++) {
                T f;
                if constexpr (kF1Lds) f = f1Lds[(16 * g + MF::rowLane(hi) + MF::rowReg(k)) * 64 + 16 * u + lo];
                else f = f1[u][g][k];
                z = MF::mma(f, d1[g][k], z);
              }
            }
#pragma unroll
          for (int k = 0; k < 4; k++) {
            T o = z[k] * alpha;
            if (HAS_Y) o += beta * yv[k];
            bufferStore(o, out, lane, (16 * u + MF::rowReg(k)) * t.Q2 * ES);
          }
        }
    }
    if (!more) return;
  }
}

bool pairAnyFits(uint32_t nf, const uint32_t* p, const uint32_t* q, uint64_t Kin) {
  if (nf != 2) return false;
  for (int j = 0; j < 2; j++) if (p[j] < 1 || p[j] > kPaMax || q[j] < 1 || q[j] > kPaMax) return false;
  return Kin == (uint64_t)p[0] * p[1];
}
bool pairAnySupported(const StepArgs& a, DType dt) {
  if (!pairAnyFits(a.nf, a.p, a.q, a.Kin) || a.batch == 0 || a.batch > 65535 || a.M == 0) return false;
  if (a.in_ldc != 1 || a.out_ldc != 1 || a.in_ldm != (int64_t)a.Kin || a.out_ldm != (int64_t)a.Kout) return false;
  if (a.Kout != (uint64_t)a.q[0] * a.q[1]) return false;
  if (a.y && (a.y_ldc != 1 || a.y_ldm != (int64_t)a.Kout)) return false;
  for (int j = 0; j < 2; j++)
    if (!(a.f_sq[j] == 1 && a.f_sp[j] == (int64_t)a.q[j]) && !(a.f_sp[j] == 1 && a.f_sq[j] == (int64_t)a.p[j])) return false;
  return true;
}

static uint32_t paWaves(int PB, uint32_t Q2) {
  const uint32_t blocks = (Q2 + 15) / 16, waves = blocks > 2 ? 4 : blocks;
  return std::max(waves, 4 / paItems(PB));
}
// (several rows per workgroup only where there are rows for all CUs twice over)
static uint32_t paRows(uint32_t waves, uint64_t rows, uint32_t cus) {
  uint32_t items = 4 / waves;
  while (items > 1 && rows < 2ull * items * cus) items /= 2;
  return items;
}
// Workgroups per batch entry: two waves per SIMD at once, four of the kernels that need few registers.
// (us, rounded up before: sgemkm 4979 x 29x29(x)49x49, 6 entries 315 -> 204, 3954 x 44^2, 3 entries 167 -> 110, dgemkm 513 x 34^2,
// 12 entries 138 -> 70)
static uint32_t paWorkgroups(int PB, size_t es, uint32_t tiles, uint32_t batch, uint32_t cus) {
  return persistentWorkgroups(tiles, batch, (es == 4 && PB == 2 ? 4 : 2) * cus);
}
PairAnyWork pairAnyWork(const uint32_t* p, const uint32_t* q, uint64_t M, uint32_t batch, DType dt, uint32_t cus) {
  const int PB = std::max(p[0], p[1]) > 32 ? 4 : 2;
  PairAnyWork w;
  w.rows = paRows(paWaves(PB, q[0]), M * batch, cus);
  const uint64_t tiles = (M + w.rows - 1) / w.rows, at = paWorkgroups(PB, dtypeSize(dt), (uint32_t)std::min<uint64_t>(tiles, UINT32_MAX), batch, cus);
  w.rounds = (tiles + at - 1) / at;
  return w;
}

template <typename T, int PB, int QB, bool HAS_Y>
static hipError_t launchPairAnyAs(const StepArgs& a, hipStream_t stream) {
  constexpr uint32_t VE = 16 / sizeof(T);
  PairAnyTile t{};
  t.P2 = a.p[0]; t.Q2 = a.q[0]; t.P1 = a.p[1]; t.Q1 = a.q[1];
  const uint32_t cus = (uint32_t)deviceCUs();
  t.waves = paWaves(PB, t.Q2);
  t.items = paRows(t.waves, (uint64_t)a.M * a.batch, cus);
  t.tiles = (a.M + t.items - 1) / t.items;
  t.pitchedMagic = t.P2 % VE == 0 && t.P2 > VE ? (uint32_t)((1ull << 32) / (t.P2 / VE)) + 1 : 0;       // (pieces are below 2^12)
  constexpr bool f1Lds = sizeof(T) == 8 && PB == 4;
  const size_t lds = t.items * t.P1 * (t.P2 + VE) * sizeof(T) + 64 + (f1Lds ? 64 * 64 * sizeof(T) : 0);
  const auto kernel = kron_pair_any_kernel<T, PB, QB, HAS_Y>;
  static PerDeviceOnce attrOnce;
  const int dev = launchDeviceIndex();
  if (lds > 65536 && !attrOnce.done(dev)) {
    if (const hipError_t e = hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024); e != hipSuccess) return e;
    attrOnce.mark(dev);
  }
  hipLaunchKernelGGL(kernel, dim3(paWorkgroups(PB, sizeof(T), t.tiles, a.batch, cus), innerEntries(a), outerEntries(a)), dim3(kPaThreads), lds, stream, a, t, a.outer);
  return hipGetLastError();
}
template <typename T, int PB, int QB>
static hipError_t launchPairAnyT(const StepArgs& a, hipStream_t stream) {
  return a.y && a.epilogue ? launchPairAnyAs<T, PB, QB, true>(a, stream) : launchPairAnyAs<T, PB, QB, false>(a, stream);
}
template <typename T>
static hipError_t launchPairAnyT(const StepArgs& a, hipStream_t stream) {
  const bool p = std::max(a.p[0], a.p[1]) > 32, q = std::max(a.q[0], a.q[1]) > 32;
  if (p) return q ? launchPairAnyT<T, 4, 4>(a, stream) : launchPairAnyT<T, 4, 2>(a, stream);
  return q ? launchPairAnyT<T, 2, 4>(a, stream) : launchPairAnyT<T, 2, 2>(a, stream);
}
hipError_t launchPairAny(const StepArgs& a, DType dt, hipStream_t stream) {
  if (!pairAnySupported(a, dt)) return hipErrorInvalidValue;
  return dt == DType::F32 ? launchPairAnyT<float>(a, stream) : launchPairAnyT<double>(a, stream);
}

}  // namespace fk
