/*
 * fastkron_ext.h -- additions of the gfx950 library that have no counterpart in the FastKron
 * reference header.  Nothing in include/fastkron.h depends on them.
 */
#pragma once
#include "fastkron.h"

#ifdef __cplusplus
extern "C" {
#endif

/*
 * Describes the launch plan of the most recent GeMKM/GeKMM call on `handle` as text:
 *   "<problem string>;<lo>-<hi>:<kernel name>;..."   (one entry per launch, in launch order)
 * Writes at most `bufLen` bytes including the terminating NUL and returns the length the full text
 * needs (excluding the NUL), or 0 when no call has been made.  Used by the benchmark to attribute
 * time to kernels and by tests to assert which kernels ran.  The reference only prints this
 * information under FASTKRON_LOG=INFO (reference src/kernel_db/kernel_db.cpp:282-285).
 */
size_t fastKronGetLastPlan(fastKronHandle handle, char* buf, size_t bufLen);

/*
 * Path of the text file tuned launch plans are loaded from and saved to (also settable with the
 * FASTKRON_TUNED_DB environment variable before fastKronInit).  NULL or "" switches persistence off.
 * The reference keeps tuning results in memory only (reference src/autotuner/autotuner.h:101-116).
 */
fastKronError fastKronSetTunedDB(fastKronHandle handle, const char* path);

/*
 * Plan-only mode (on != 0): GeMKM/GeKMM calls on `handle` run every argument check, the launch planner and each
 * chosen kernel's check of the concrete buffers (alignment, strides), but launch nothing and touch no device;
 * an MI355X is assumed when none has been initialised.  fastKronGetLastPlan then names the kernels and
 * fastKronGetLastLaunches lists the launches the call would have made, one text line per launch:
 *   "kernel=<name> lo=<lo> hi=<hi> M=<rows> batch=<n> Kin=<cols> Kout=<cols> in=<ptr> out=<ptr> y=<ptr>
 *    in_batch=<elems> out_batch=<elems> y_batch=<elems> stream_in=<0|1> stream_out=<0|1> f_batch=<elems>,<elems>,..."
 * with " inner=<n> outer_in=<elems> outer_out=<elems> outer_y=<elems>" behind it for two batch dimensions (batch entry b is
 * entry b % inner of the first and b / inner of the second).
 * fastKronGradForward is such a call; for fastKronGradBackward the lines are kernel=gradient_step, one per step of the chain,
 * and kernel=gradient_sum.
 * Meant for host-side tests of the planner and for inspecting what a call will do.  The reference has no such
 * mode; its nearest counterpart is the kernel series printed under FASTKRON_LOG=INFO
 * (reference src/kernel_db/kernel_db.cpp:282-285).
 */
fastKronError fastKronSetPlanOnly(fastKronHandle handle, int on);
size_t fastKronGetLastLaunches(fastKronHandle handle, char* buf, size_t bufLen);

/*
 * sgemkm for callers that cannot allocate device memory: code under HIP graph capture, tight serving loops,
 * harnesses that forbid hipMalloc.  It has no counterpart in the reference.  Same arguments and result as sgemkm
 * (include/fastkron.h) without temp1 / temp2: the two temporaries and the workspace for merged factors are parts of
 * one array that the library keeps in device memory on every GPU it is loaded on, for the life of the process
 * (2 * FASTKRON_STATIC_SCRATCH_TEMP_BYTES + 512 KiB).  The call itself allocates and frees nothing and never tunes.
 * A problem whose temporaries (gekmmSizes' tmpElems * 4 bytes) exceed FASTKRON_STATIC_SCRATCH_TEMP_BYTES is refused
 * with fastKronInvalidArgument and a message on stderr.  All calls on one GPU share the array: calls that overlap
 * on one GPU race, whatever their handles and streams.  fastKronInitHIP resolves the array's address on its GPU.
 */
#define FASTKRON_STATIC_SCRATCH_TEMP_BYTES (16u << 20)
fastKronError sgemkmStaticScratch(fastKronHandle handle, fastKronBackend backend, uint32_t M, uint32_t N,
                                  uint32_t Ps[], uint32_t Qs[], const float* X, fastKronOp opX,
                                  const float* const Fs[], fastKronOp opFs, float* Z, float alpha, float beta,
                                  const float* Y);

/*
 * Kernels whose workgroups wait for each other inside one launch (the two-phase 4x4^6 GeKMM kernel) keep their counters
 * in device memory of the handle and bound every wait; a wait that runs out sets an error word there and the results
 * of that launch are not valid.  fastKronGetSyncError synchronises the handle's stream, copies the word to *word
 * (0: no wait ever ran out) and clears it.  fastKronSetSyncHelpAfter sets, for every handle of the process, after how
 * many polls a waiting workgroup runs the missing work of others itself (default 100000, far beyond what a launch
 * needs when all its workgroups run; 0 makes every workgroup do so at once, which tests use to cover that path).
 * Neither has a counterpart in the reference, whose kernels never synchronise across workgroups.
 */
fastKronError fastKronGetSyncError(fastKronHandle handle, uint32_t* word);
fastKronError fastKronSetSyncHelpAfter(uint32_t polls);

/*
 * Measurement aid, no counterpart in the reference: launches on the handle's stream a copy kernel Z = 1.5 X + 0.5 Y over
 * 4096 x M fp32 matrices (M a multiple of 2048, at most 16384) that touches memory the way one of the 4x4^6 GeKMM kernels
 * does and computes nothing else.  pattern 0: contiguous 16-byte accesses; 1: 32-byte strips of 8 columns, all 4096
 * rows per workgroup; 2: 256-byte pieces in two phases with an intermediate T (4096 x M floats) passed through the
 * L2 and workgroups waiting for each other.  `python bench.py --pattern-ceilings` times them beside the kernels.
 */
fastKronError fastKronProbeCopyPattern(fastKronHandle handle, int pattern, const float* X, const float* Y, float* Z,
                                       float* T, uint32_t M);

/*
 * A product with two batch dimensions of which the factors have the second one only (X of shape (a, 1), factors of shape
 * (b) ...): entry (o, i) of count[0] x count[1] takes X at o * strideX[0] + i * strideX[1] elements, the i-th factors (P*Q
 * elements apart) and Y and Z likewise.  mkm, dbl as below; the temporaries hold count[0] * count[1] entries of the size that
 * gekmmSizes gives.  Results are those of count[0] strided-batched calls.  (The reference loops over outer batch dimensions
 * in Python, reference pyfastkron/fastkronbase.py:104-518.)
 */
fastKronError fastKronProductOuter(fastKronHandle handle, int mkm, int dbl, uint32_t M, uint32_t N, const uint32_t Ps[], const uint32_t Qs[],
                                   const void* X, fastKronOp opX, const uint64_t strideX[2], const void* const Fs[], fastKronOp opFs, void* Z,
                                   const uint64_t strideZ[2], double alpha, double beta, const uint32_t count[2], const void* Y,
                                   const uint64_t strideY[2], void* temp1, void* temp2);

/*
 * Gradients.  fastKronGradForward computes Z like the forward family of include/fastkron.h (alpha = 1, no Y) and keeps in
 * `save` what the backward pass needs; fastKronGradBackward takes the gradient gZ of Z (laid out like Z, batch entries
 * one after the other) and writes the gradient of X to gX (row-major M x K for MKM, K x M for KMM, one per batch entry,
 * also when X is shared by the batch) unless gX is NULL, and the gradient of every factor whose entry of gFs is not
 * NULL (row-major P x Q for MKM, Q x P for KMM whatever opFs; with perBatchFs one per batch entry, otherwise one, summed
 * over the batch).  Equal calls give equal bits.
 * mkm: 1 for Z = X (F_0 x ...), 0 for Z = (F_0 x ...) X; dbl: 0 for float, 1 for double operands.  A batch has batchCount
 * entries; X's are strideX elements apart (0: shared), the factors' P*Q elements (perBatchFs) or shared, Z's M*L.
 * fastKronGradSizes gives the elements of `save` (kept from the forward to the backward pass, with the same shapes) and
 * of `work` (scratch of the backward pass).  Both calls run on the handle's stream, allocate nothing and never synchronise.
 * The reference has the forward family only and leaves gradients to PyTorch (reference pyfastkron/fastkrontorch.py:160-217).
 */
fastKronError fastKronGradSizes(fastKronHandle handle, int mkm, int dbl, uint32_t M, uint32_t N, const uint32_t Ps[],
                                const uint32_t Qs[], fastKronOp opX, uint64_t strideX, int perBatchFs, uint32_t batchCount,
                                size_t* saveElems, size_t* workElems);
fastKronError fastKronGradForward(fastKronHandle handle, int mkm, int dbl, uint32_t M, uint32_t N, const uint32_t Ps[],
                                  const uint32_t Qs[], const void* X, fastKronOp opX, uint64_t strideX, const void* const Fs[],
                                  fastKronOp opFs, int perBatchFs, uint32_t batchCount, void* Z, void* save);
fastKronError fastKronGradBackward(fastKronHandle handle, int mkm, int dbl, uint32_t M, uint32_t N, const uint32_t Ps[],
                                   const uint32_t Qs[], const void* X, fastKronOp opX, uint64_t strideX, const void* const Fs[],
                                   fastKronOp opFs, int perBatchFs, uint32_t batchCount, const void* gZ, void* save, void* gX,
                                   void* const gFs[], void* work);
/*
 * A part of the backward pass, for callers that compute the gradient of some step's input by a product of their own: the
 * steps of the factors first .. last (fastKronGradBackward: 0 .. N-1).  gOut is the gradient of the output of the step of
 * factor `first` (gZ for 0), gIn receives the gradient of the input of the step of factor `last` (gX for N-1) unless it is
 * NULL; both are M x columns (MKM) or columns x M (KMM), batch entries one after the other.  Entries of gFs outside the
 * range are not looked at.
 */
fastKronError fastKronGradBackwardSteps(fastKronHandle handle, int mkm, int dbl, uint32_t M, uint32_t N, const uint32_t Ps[],
                                        const uint32_t Qs[], const void* X, fastKronOp opX, uint64_t strideX, const void* const Fs[],
                                        fastKronOp opFs, int perBatchFs, uint32_t batchCount, uint32_t first, uint32_t last,
                                        const void* gOut, void* save, void* gIn, void* const gFs[], void* work);

#ifdef __cplusplus
}
#endif
