// Gradients of a GeMKM / GeKMM: a forward pass that keeps every step's input and a backward pass that goes through the
// steps in the opposite order, one launch per step for the gradients of the step's input and of its factor
// (kernels/gradient_mfma.hip), one launch that adds the partial sums of all factors that have several.
//
// Every factor keeps a step of its own: merged to products of up to 64x64, chains of small factors took fewer launches
// (dgekmm 8x8^5 x 16 nine instead of eleven, 125 against 134 us), but Z and the gradient of X came out with twice the
// rounding error (8x8^4 in fp32 2.0e-7 against 1.1e-7).
// The reference chains PyTorch matmuls through the intermediates of its forward family, one factor at a time
// (reference pyfastkron/fastkrontorch.py:160-217).
#include "handle.h"

#include <algorithm>
#include <cstdio>
#include <cstring>

#include "kernels/gradient.h"
#include "kernels/launch.h"

namespace fk {

namespace {

constexpr uint64_t kMaxRows = (1ull << 31) - 16;       // rows per launch of the step kernel
constexpr uint32_t kMaxGridBatch = 65535;

size_t roundUp(size_t v) { return (v + 63) & ~(size_t)63; }       // elements: 256-byte (fp32) boundaries and better

// The chain as the two passes run it.
struct GradPlan {
  KronProblem q;                    // MKM or KMM, op(X) = N; F, X, Z, inter not set
  bool pMajor;                      // storage of the factors: element (p, q) at p*Q + q
  bool outTransposed;               // gradients of the factors are Q x P (KMM)
  bool copyX;                       // op(X) = T: each pass reads a transposed copy of X, which is not kept between them
  uint32_t xBatch;                  // entries of that copy
  // offsets into `save`, in elements
  size_t saveI[kMaxFactors], saveTotal;
  // offsets into `work`
  size_t workX, workG[2], workP[kMaxFactors], workTotal;
  uint32_t parts[kMaxFactors];      // partial sums of factor g per batch entry
};

// Row ranges of at most kMaxRows of a step: calls f(first o, count of o, first t, count of t).
template <typename F> void forRowChunks(uint64_t O, uint64_t Tn, F f) {
  if (Tn > kMaxRows) {
    for (uint64_t o = 0; o < O; o++)
      for (uint64_t t = 0; t < Tn; t += kMaxRows) f(o, (uint64_t)1, t, std::min(kMaxRows, Tn - t));
    return;
  }
  const uint64_t per = std::max<uint64_t>(1, kMaxRows / Tn);
  for (uint64_t o = 0; o < O; o += per) f(o, std::min(per, O - o), (uint64_t)0, Tn);
}

struct StepShape { uint64_t O, Tn; };               // rows u = o*Tn + t
StepShape stepShape(const KronProblem& q, uint32_t g) {
  const uint64_t S = q.colsBefore(g) / q.P[g];
  return q.mm == MMType::MKM ? StepShape{q.M, S} : StepShape{S, q.M};
}

fastKronError makePlan(const Handle::GradProblem& p, GradPlan* gp) {
  if (p.N == 0 || p.N > kMaxFactors || p.M == 0 || p.batch == 0 || !p.P || !p.Q) return fastKronInvalidKMMProblem;
  KronProblem& q = gp->q;
  q = KronProblem{};
  q.mm = p.mm; q.dt = p.dt; q.M = p.M; q.N = p.N; q.batch = p.batch;
  for (uint32_t i = 0; i < p.N; i++) {
    if (p.P[i] == 0 || p.Q[i] == 0) return fastKronInvalidKMMProblem;
    q.P[i] = p.P[i]; q.Q[i] = p.Q[i];
  }
  q.opX = fastKronOp_N; q.opF = p.opF;
  gp->pMajor = (p.mm == MMType::MKM) == (p.opF == fastKronOp_N);
  gp->outTransposed = p.mm == MMType::KMM;
  gp->copyX = p.opX == fastKronOp_T && p.M > 1;
  gp->xBatch = (p.batch > 1 && p.strideX != 0) ? p.batch : 1;
  if (q.mm == MMType::KMM && q.M == 1) {
    // a single column is the MKM of the same vector with transposed factors
    q.mm = MMType::MKM;
    q.opF = p.opF == fastKronOp_N ? fastKronOp_T : fastKronOp_N;
  }
  const uint64_t K = q.K();
  // batches against shared factors are more rows of one problem (MKM)
  if (q.mm == MMType::MKM && q.batch > 1 && !p.perBatchF && p.strideX != 0 && (p.strideX == q.M * K || gp->copyX) &&
      (uint64_t)q.M * q.batch < (1ull << 32)) {
    q.M *= q.batch; q.batch = 1;
  }
  const size_t nb = q.batch;
  size_t off = 0;
  auto take = [&](size_t elems) { const size_t o = off; off += roundUp(elems); return o; };
  for (uint32_t g = 1; g < q.N; g++) gp->saveI[g] = take(nb * q.M * q.colsAfter(g));      // output of step g
  gp->saveTotal = off;
  off = 0;
  gp->workX = gp->copyX ? take((size_t)gp->xBatch * p.M * K) : 0;
  size_t widest = 0;
  for (uint32_t g = 0; g + 1 < q.N; g++) widest = std::max<size_t>(widest, q.colsBefore(g));
  for (int i = 0; i < 2; i++) gp->workG[i] = q.N > 1u + i ? take(nb * q.M * widest) : 0;
  for (uint32_t g = 0; g < q.N; g++) {
    const StepShape s = stepShape(q, g);
    uint32_t parts = 0;
    forRowChunks(s.O, s.Tn, [&](uint64_t, uint64_t on, uint64_t, uint64_t tn) { parts += gradWorkgroups(q.P[g], q.Q[g], on * tn, q.batch); });
    gp->parts[g] = parts;
    gp->workP[g] = take(nb * parts * q.P[g] * q.Q[g]);
  }
  gp->workTotal = off;
  return fastKronSuccess;
}

}  // namespace

fastKronError Handle::gradSizes(const GradProblem& p, size_t* saveElems, size_t* workElems) const {
  if (!saveElems || !workElems) return fastKronInvalidArgument;
  GradPlan gp;
  fastKronError e = makePlan(p, &gp);
  if (e != fastKronSuccess) return e;
  *saveElems = gp.saveTotal; *workElems = gp.workTotal;
  return fastKronSuccess;
}

// X (op T) of every batch entry with a stride of its own, transposed to `to`.
hipError_t Handle::transposeX(const GradProblem& p, void* to) {
  KronProblem t{};
  t.mm = p.mm; t.dt = p.dt; t.M = p.M; t.N = p.N; t.batch = p.batch; t.X = p.X; t.strideX = p.strideX;
  for (uint32_t i = 0; i < p.N; i++) { t.P[i] = p.P[i]; t.Q[i] = p.Q[i]; }
  return launchTransposeX(t, to, (uint64_t)p.M * t.K());
}

fastKronError Handle::gradForward(const GradProblem& p, void* Z, void* save) {
  if (!Z || !p.X || !p.F) return fastKronInvalidArgument;
  for (uint32_t i = 0; i < p.N; i++) if (!p.F[i]) return fastKronInvalidKMMProblem;
  GradPlan gp;
  fastKronError e = makePlan(p, &gp);
  if (e != fastKronSuccess) return e;
  if (gp.saveTotal && !save) return fastKronInvalidArgument;
  e = planOnly_ ? fastKronSuccess : ensureDevice();
  if (e != fastKronSuccess) return e;
  launchLog_.clear();
  const size_t es = dtypeSize(p.dt);
  char* sv = (char*)save;
  KronProblem q = gp.q;
  q.X = p.X; q.strideX = q.batch > 1 ? p.strideX : 0;
  if (gp.copyX) {
    // (a first factor beyond the padded step, which the plain kernel runs, is ahead on X as it is stored in the MKM layout: its
    // lanes then lie along neighbours, sgemkm 200 x 320x320^2 with all gradients 2.7 ms against 3.8; in the KMM layout they
    // do so on the copy, sgekmm 8x8 (x) 300x300 x 4166 0.78 against 1.02)
    const bool plainFirst = q.mm == MMType::MKM && (q.P[q.N - 1] > 256 || q.Q[q.N - 1] > 512);
    if (q.N > 1 && !plainFirst && (uint64_t)gp.xBatch * p.M * q.K() <= (uint64_t)q.batch * q.M * q.L()) {
      // the copy stands in Z, which only the last of the launches writes
      if (!planOnly_ && transposeX(p, Z) != hipSuccess) return fastKronInvalidArgument;
      q.X = Z; q.strideX = q.batch > 1 && gp.xBatch > 1 ? (uint64_t)p.M * q.K() : 0;
      q.xJustWritten = true;
    } else {
      // the first launch reads X as it is stored (entry by entry: not as rows of one problem)
      q.M = p.M; q.batch = p.batch;
      q.opX = fastKronOp_T; q.strideX = q.batch > 1 ? p.strideX : 0;
    }
  }
  for (uint32_t g = 0; g < q.N; g++) {
    q.strideF[g] = p.perBatchF && q.batch > 1 ? (uint64_t)q.P[g] * q.Q[g] : 0;
    q.F[g] = p.F[g];
  }
  q.forward = true; q.strided = q.batch > 1; q.haveStrideInter = true;
  for (uint32_t g = 1; g < q.N; g++) {
    q.inter[g - 1] = sv + gp.saveI[g] * es;
    q.strideInter[g - 1] = (uint64_t)q.M * q.colsAfter(g);
  }
  q.Z = Z; q.strideZ = q.batch > 1 ? (uint64_t)q.M * q.L() : 0;
  q.alpha = 1.0; q.beta = 0.0;
  callWs_ = false;
  return runOnline(q, nullptr, nullptr, nullptr);
}

fastKronError Handle::gradBackward(const GradProblem& p, uint32_t first, uint32_t last, const void* gOut, void* save, void* gIn, void* const* gF,
                                   void* work) {
  if (!gOut || !p.X || !p.F || !gF || first > last || last >= p.N) return fastKronInvalidArgument;
  for (uint32_t i = 0; i < p.N; i++) if (!p.F[i]) return fastKronInvalidKMMProblem;
  GradPlan gp;
  fastKronError e = makePlan(p, &gp);
  if (e != fastKronSuccess) return e;
  if ((gp.saveTotal && !save) || (gp.workTotal && !work)) return fastKronInvalidArgument;
  e = planOnly_ ? fastKronSuccess : ensureDevice();
  if (e != fastKronSuccess) return e;
  launchLog_.clear();
  const KronProblem& q = gp.q;
  const size_t es = dtypeSize(p.dt);
  const uint32_t ve = (uint32_t)(16 / es);
  char* sv = (char*)save;
  char* wk = (char*)work;
  const bool mkm = q.mm == MMType::MKM;
  // the last factor (in chain order) whose gradient is wanted: nothing behind it is computed unless gIn is
  int lastWanted = -1;
  bool wanted[kMaxFactors] = {};
  for (uint32_t g = first; g <= last; g++) {
    wanted[g] = gF[g] != nullptr;
    if (wanted[g]) lastWanted = (int)g;
  }
  if (gIn) lastWanted = (int)last;
  if (gp.copyX && wanted[q.N - 1] && !planOnly_ && transposeX(p, wk + gp.workX * es) != hipSuccess) return fastKronInvalidArgument;

  const void* g = gOut;
  uint64_t gBatch = q.batch > 1 ? (uint64_t)q.M * q.colsAfter(first) : 0;
  for (int i = (int)first; i <= lastWanted; i++) {
    const uint64_t Kin = q.colsBefore(i), S = Kin / q.P[i];
    const bool lastStep = i + 1 == (int)q.N;
    GradStepArgs a{};
    a.P = q.P[i]; a.Q = q.Q[i];
    const char* F = (const char*)p.F[i];
    a.f_sp = gp.pMajor ? (int64_t)a.Q : 1;
    a.f_sq = gp.pMajor ? 1 : (int64_t)a.P;
    a.f_batch = p.perBatchF && q.batch > 1 ? (uint64_t)a.P * a.Q : 0;
    const char* in; uint64_t inBatch;
    if (lastStep) {
      in = gp.copyX ? wk + gp.workX * es : (const char*)p.X;
      inBatch = q.batch > 1 ? (gp.copyX ? (gp.xBatch > 1 ? (uint64_t)q.M * Kin : 0) : p.strideX) : 0;
    } else {
      in = sv + gp.saveI[i + 1] * es;
      inBatch = (uint64_t)q.M * Kin;
    }
    void* gin = nullptr;
    if (i == (int)last) gin = gIn;
    else if (i < lastWanted) gin = wk + gp.workG[i & 1] * es;
    const uint64_t ginBatch = (uint64_t)q.M * Kin;
    if (mkm) {
      a.in_o = (int64_t)Kin; a.in_t = a.P; a.in_p = 1;
      a.g_o = (int64_t)(S * a.Q); a.g_t = 1; a.g_q = (int64_t)S;
    } else {
      a.in_o = (int64_t)a.P * q.M; a.in_t = 1; a.in_p = q.M;
      a.g_o = q.M; a.g_t = 1; a.g_q = (int64_t)(S * q.M);
    }
    a.in_batch = inBatch; a.g_batch = gBatch; a.gin_batch = ginBatch;
    if (!wanted[i] && !gin) { g = gin; gBatch = ginBatch; continue; }
    // a single partial sum is the gradient: written where it goes (2048x2048, 7 rows: the launch that adds them took 38 us to
    // copy it, the step itself 10)
    const bool direct = wanted[i] && gp.parts[i] == 1 && (p.perBatchF || q.batch == 1);
    a.partSp = direct && gp.outTransposed ? 1 : a.Q;
    a.partSq = direct && gp.outTransposed ? a.P : 1;
    char* partials = direct ? (char*)gF[i] : wk + gp.workP[i] * es;
    const StepShape sh = stepShape(q, i);
    uint32_t partFirst = 0;
    hipError_t he = hipSuccess;
    forRowChunks(sh.O, sh.Tn, [&](uint64_t o0, uint64_t on, uint64_t t0, uint64_t tn) {
      GradStepArgs c = a;
      const int64_t inOff = (int64_t)o0 * a.in_o + (int64_t)t0 * a.in_t, gOff = (int64_t)o0 * a.g_o + (int64_t)t0 * a.g_t;
      c.Tn = (uint32_t)tn; c.U = (uint32_t)(on * tn);
      if (tn > 1) {
        uint32_t s = 0;
        while ((1ull << s) < tn) s++;
        c.tnShift = 31 + s;
        c.tnMagic = ((1ull << c.tnShift) / tn) + 1;
      }
      c.gridX = gradWorkgroups(c.P, c.Q, c.U, q.batch);
      c.partStride = gp.parts[i]; c.partFirst = partFirst;
      partFirst += c.gridX;
      for (uint32_t b0 = 0; b0 < q.batch && he == hipSuccess; b0 += kMaxGridBatch) {
        c.batch = std::min(q.batch - b0, kMaxGridBatch);
        c.in = in + ((size_t)b0 * inBatch + inOff) * es;
        c.g = (const char*)g + ((size_t)b0 * gBatch + gOff) * es;
        c.gin = gin ? (char*)gin + ((size_t)b0 * ginBatch + inOff) * es : nullptr;
        c.f = F + (size_t)b0 * a.f_batch * es;
        c.partial = wanted[i] ? partials + (size_t)b0 * gp.parts[i] * c.P * c.Q * es : nullptr;
        auto aligned = [&](const void* ptr, int64_t s1, int64_t s2, uint64_t sb) {
          return (uintptr_t)ptr % 16 == 0 && s1 % ve == 0 && s2 % ve == 0 && sb % ve == 0;
        };
        const bool t4 = tn % 4 == 0;
        c.vecG = t4 && aligned(c.g, c.g_o, c.g_q, gBatch);
        c.vecIn = t4 && c.in_t == 1 && aligned(c.in, c.in_o, c.in_p, inBatch);
        c.vecOut = c.gin && c.in_p == 1 && c.P % 4 == 0 && aligned(c.gin, c.in_o, c.in_t, ginBatch);
        if (planOnly_) {
          char line[192];
          const int n = snprintf(line, sizeof(line), "kernel=gradient_step lo=%d hi=%d rows=%u batch=%u sums=%u in=%p g=%p gin=%p partial=%p\n", i, i, c.U,
                                 c.batch, c.gridX, c.in, c.g, c.gin, c.partial);
          launchLog_.append(line, n > 0 ? (size_t)n : 0);
        } else he = launchGradStep(c, p.dt, stream_);
      }
    });
    if (he != hipSuccess) return fastKronInvalidArgument;
    g = gin; gBatch = ginBatch;
  }

  // sum the partial sums of all factors
  GradReduceArgs ra{};
  const uint32_t fBatch = p.perBatchF ? q.batch : 1;
  auto reduceNow = [&]() -> hipError_t {
    for (uint32_t b0 = 0; b0 < fBatch && ra.count; b0 += kMaxGridBatch) {
      GradReduceArgs c = ra;
      for (uint32_t i = 0; i < c.count; i++) {
        const size_t pq = (size_t)c.r[i].P * c.r[i].Q;
        c.r[i].partial = (const char*)c.r[i].partial + (size_t)b0 * c.r[i].count * pq * es;
        c.r[i].out = (char*)c.r[i].out + (size_t)b0 * pq * es;
      }
      const uint32_t n = std::min(fBatch - b0, kMaxGridBatch);
      if (planOnly_) launchLog_ += "kernel=gradient_sum factors=" + std::to_string(c.count) + " batch=" + std::to_string(n) + "\n";
      else if (const hipError_t he = launchGradReduce(c, n, p.dt, stream_); he != hipSuccess) return he;
    }
    ra.count = 0;
    return hipSuccess;
  };
  for (int i = (int)first; i <= lastWanted; i++) {
    if (!wanted[i] || (gp.parts[i] == 1 && (p.perBatchF || q.batch == 1))) continue;
    GradReduce& r = ra.r[ra.count++];
    r.P = q.P[i]; r.Q = q.Q[i];
    r.count = gp.parts[i] * (p.perBatchF ? 1 : q.batch);
    r.partial = wk + gp.workP[i] * es;
    r.out = gF[i];
    r.osp = gp.outTransposed ? 1 : r.Q; r.osq = gp.outTransposed ? r.P : 1;
    if (ra.count == kMaxGradReduce && reduceNow() != hipSuccess) return fastKronInvalidArgument;
  }
  if (reduceNow() != hipSuccess) return fastKronInvalidArgument;
  return fastKronSuccess;
}

}  // namespace fk
