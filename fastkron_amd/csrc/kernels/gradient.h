// Launch arguments of the backward-pass kernels (gradient_mfma.hip).
#pragma once
#include <hip/hip_runtime.h>
#include "../problem.h"

namespace fk {

// One step's backward pass.  Row u = o*Tn + t of the step's input: element p at in + o*in_o + t*in_t + p*in_p; of its
// output gradient: element q at g + o*g_o + t*g_t + q*g_q.  gin has the strides of `in`.
struct GradStepArgs {
  const void* in; const void* g; void* gin; void* partial;     // gin / partial null: not wanted
  const void* f; int64_t f_sp, f_sq;
  uint64_t in_batch, g_batch, gin_batch, f_batch;
  int64_t in_o, in_t, in_p, g_o, g_t, g_q;
  uint32_t P, Q, Tn, U, batch;                                 // U rows per batch entry, below 2^31
  uint64_t tnMagic; uint32_t tnShift;                          // u / Tn = (u * tnMagic) >> tnShift (tnMagic 0: Tn = 1)
  uint32_t vecIn, vecG, vecOut;                                // 16-byte accesses possible (alignment and Tn, P multiples of 4)
  uint32_t gridX;                                              // workgroups along u = partial sums of this launch
  uint32_t partStride, partFirst;                              // partial sums per batch entry, first one of this launch
  uint32_t partSp, partSq;                                     // element (p, q) of a partial sum at p*partSp + q*partSq
  uint32_t qChunks, fPitch;                                    // set by the launcher
};

struct GradReduce {
  const void* partial; void* out;
  uint32_t P, Q, count;                                        // partial sums per entry of grid z
  uint32_t osp, osq;                                           // element (p, q) of the result at out + p*osp + q*osq
};
constexpr uint32_t kMaxGradReduce = 32;
struct GradReduceArgs { GradReduce r[kMaxGradReduce]; uint32_t count; };

constexpr size_t kGradLdsMax = 140 * 1024;

// Workgroups (partial sums) a step is given.
uint32_t gradWorkgroups(uint32_t P, uint32_t Q, uint64_t U, uint32_t batch);
hipError_t launchGradStep(const GradStepArgs& a, DType dt, hipStream_t stream);
hipError_t launchGradReduce(const GradReduceArgs& a, uint32_t batch, DType dt, hipStream_t stream);

}  // namespace fk
